"""CPU-only check of csrc/fmha_items.h: no access of a workgroup's list of work items lies in the same stretch between two barriers as a write
that would change what it sees."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "understanding-gpu-architecture-implications-on-llm-serving-workloads_amd", "csrc")

# Iteration n of the loop over the items, as the kernel orders it. Behind the last barrier of iteration n - 1 every wave reads item n - 1, the
# last wave goes on and writes the items from n on (if it is time to), then all meet at the first barrier of iteration n, behind which
# item n is read. Between two barriers a slow wave's read may come before or after the last wave's writes: it has to find its item either way.
PROGRAM = """
#include <cstdio>
#include "fmha_items.h"
using mi355::ListedItems;
int main() {
    int held[ListedItems::kHeld];
    for (int& h : held) h = -1;
    for (int n = 1; n <= 5 * ListedItems::kHeld + 3; ++n) {
        if (n > 1 && held[ListedItems::entry(n - 1)] != n - 1) { printf("item %d is not there\\n", n - 1); return 1; }
        if (ListedItems::refill(n))
            for (int lane = 0; lane < ListedItems::kAtOnce; ++lane) held[ListedItems::entry(n + lane)] = n + lane;
        if (n > 1 && held[ListedItems::entry(n - 1)] != n - 1) { printf("item %d is overwritten while it is read\\n", n - 1); return 1; }
        if (held[ListedItems::entry(n)] != n) { printf("item %d was not written\\n", n); return 1; }
    }
    return 0;
}
"""


def run(tmp_path, edit=lambda header: header):
    cxx = os.environ.get("CXX", "g++")
    if shutil.which(cxx) is None:
        pytest.skip("no C++ compiler here")
    (tmp_path / "fmha_items.h").write_text(edit(open(os.path.join(CSRC, "fmha_items.h")).read()))
    (tmp_path / "order.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "order.cpp", "-o", "order"], cwd=tmp_path, check=True)
    return subprocess.run([str(tmp_path / "order")], stdout=subprocess.PIPE, text=True)


def test_no_listed_item_is_overwritten_while_a_wave_may_still_read_it(tmp_path):
    done = run(tmp_path)
    assert done.returncode == 0, done.stdout


def test_the_check_finds_a_list_of_one_half(tmp_path):
    done = run(tmp_path, lambda header: header.replace("kHeld = 2 * kAtOnce", "kHeld = kAtOnce"))
    assert done.returncode == 1 and done.stdout == "item 64 is overwritten while it is read\n"
