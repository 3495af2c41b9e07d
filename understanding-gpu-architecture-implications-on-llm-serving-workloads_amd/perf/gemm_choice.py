"""How good the library's choice of a GEMM kernel is: times the kernel that a product takes by itself against every pinned kernel
(variants of mi355_internal_hgemm_variant) over products drawn with a fixed seed, second operands cycling through more
memory than the caches hold, and prints the regret: time of the choice over that of the fastest kernel.

    python perf/gemm_choice.py [--products 200] [--seed 1] [--rows 8192] [--list 20]
"""
import argparse
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import mi355_serving as lib  # noqa: E402

TILE = {1: (256, 256), 2: (128, 128), 3: (64, 128), 4: (64, 64), 5: (128, 256), 6: (256, 128), 7: (32, 64), 9: (64, 64)}
RANGES = (2, 3, 4, 5, 6, 8, 10, 12, 16)


def variants(M, N, K, layout):
    """The pinned kernels that fit a product, ranges of K included."""
    out = [8] if M <= 64 else []
    if M <= 16 and layout != "NT":      # 128 columns and ranges of K
        out += [8 + 16 * s for s in (2, 4, 6, 8) if s * 256 <= K]
    for shape, (bm, bn) in TILE.items():
        if (shape == 7 and layout == "TN") or (shape == 9 and M > 64) or (bm > 64 and bm >= 2 * M):
            continue
        bm, bn = (bn, bm) if shape == 3 and layout == "NT" else (bm, bn)
        tiles = -(-M // bm) * -(-N // bn)
        out.append(shape)
        for s in RANGES:
            if shape == 9 or tiles > 400 or tiles * s > 1200 or -(-K // 64) < 2 * s or tiles * s * bm * bn > 16 << 20:
                break
            out += [shape + 16 * s + 4096] + [shape + 16 * s] * (shape != 1)      # 256x256 tiles have the merge kernel only
    return out


def draw(rng, rows):
    log = lambda lo, hi: int(round(lo * (hi / lo) ** rng.random()))
    while True:
        M, N, K, layout = log(1, rows), log(128, 131072), log(128, 14336), rng.choice(("NN", "NT", "TN"))
        step = 64 if rng.random() < 0.6 else 8
        N, K = max(step, N // step * step), max(step, K // step * step)
        if M * N * K <= 2.5e11 and N * K <= 5e8 and M * (N + K) <= 2e8:
            return M, N, K, layout


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--products", type=int, default=200)
    ap.add_argument("--seed", type=int, default=1)
    ap.add_argument("--rows", type=int, default=8192)
    ap.add_argument("--list", type=int, default=20, help="products with the largest regret to print")
    args = ap.parse_args()
    rng, cdll = random.Random(args.seed), lib.load()
    pool = torch.randn(1 << 26, device="cuda").mul_(0.05).half().repeat(16)      # 2 GiB of operands
    c = torch.empty(1 << 28, dtype=torch.float16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

    def time_us(M, N, K, layout, variant, n):
        lda, ldb = ((M + 7) // 8 * 8 if layout == "TN" else K), (K if layout == "NT" else N)
        a_elems = (K if layout == "TN" else M) * lda
        b_first, b_elems = -(-a_elems // 128) * 128, -(-(N * K) // 128) * 128
        copies = max(1, min(64, (pool.numel() - b_first) // b_elems, -(-(200 << 20) // b_elems)))
        calls = [(pool.data_ptr(), pool.data_ptr() + 2 * (b_first + i * b_elems), c.data_ptr(), M, N, K, lda, ldb, N, lib.LAYOUTS[layout],
                  lib.DTYPE_FP16, variant, stream) for i in range(copies)]
        begin.record()
        for i in range(n):
            rc = cdll.mi355_internal_hgemm_variant(*calls[i % copies])
            assert rc == 0, (M, N, K, layout, variant, rc)
        end.record()
        end.synchronize()
        return begin.elapsed_time(end) * 1e3 / n

    rows = []
    for i in range(args.products):
        M, N, K, layout = draw(rng, args.rows)
        chosen = cdll.mi355_internal_hgemm_choice(M, N, K, K if layout == "NT" else N, lib.LAYOUTS[layout], None)
        if chosen == 8 and layout != "NT":
            chosen += 16 * cdll.mi355_internal_hgemm_wide_ranges(M, N, K, N, lib.LAYOUTS[layout])
        todo = sorted(set(variants(M, N, K, layout)) | {chosen})
        best = {v: time_us(M, N, K, layout, v, 4) for v in todo}
        for _ in range(3):
            for v in todo:
                if v == chosen or best[v] < 1.5 * min(best.values()):
                    best[v] = min(best[v], time_us(M, N, K, layout, v, max(5, min(100, int(800 / best[v])))))
        fastest = min(best, key=best.get)
        rows.append((best[chosen] / best[fastest], M, N, K, layout, chosen, best[chosen], fastest, best[fastest]))
        if i % 50 == 49:
            print("%d products" % (i + 1), flush=True)
    rows.sort(reverse=True)
    regret = [r[0] for r in rows]
    print("choice / fastest kernel over %d products: mean %.3f, 90 %% of them below %.3f, %d above 1.05, %d above 1.10" % (
        len(rows), math.exp(sum(map(math.log, regret)) / len(rows)), sorted(regret)[int(0.9 * len(rows))],
        sum(r > 1.05 for r in regret), sum(r > 1.10 for r in regret)))
    for r in rows[:args.list]:
        print("  %.2f  %5d x %6d x %5d %s  chosen %4d %7.1f us   fastest %4d %7.1f us" % r)


if __name__ == "__main__":
    main()
