"""The store of what is prepared per weight (HELLM/BoundedStore.hpp): the bound is on the sum of the costs, the oldest goes first, an entry put again
counts once and becomes the newest, one beyond the limit is kept alone."""
import os
import subprocess

HOST = os.path.join(os.path.dirname(__file__), "..", "encryption-friendly_llm_architecture_amd", "csrc", "host")
PROGRAM = r"""
#include <cstdio>
#include <memory>
#include "HELLM/BoundedStore.hpp"
typedef HELLM::BoundedStore<int, std::unique_ptr<int>> Store;
static void show(const Store &s) {
    for (int k = 0; k < 10; k++)
        if (auto *e = s.find(k)) std::printf("%d:%d ", k, **e);
    std::printf("= %d\n", (int)s.cost());
}
int main() {
    Store s(10);
    auto put = [&](int k, int v, int cost) { if (*s.keep(k, std::make_unique<int>(v), cost) != v) std::printf("wrong "); show(s); };
    put(0, 100, 4); put(1, 101, 4); put(2, 102, 2);   // exactly full
    put(3, 103, 1);                                    // the oldest goes
    put(1, 111, 3); put(4, 104, 5);                    // put again: the newest of its kind; 2 goes, then fits
    s.makeRoom(5); show(s);
    put(5, 105, 25); put(6, 106, 1);
    s.clear(); show(s);
    put(7, 107, 10);
}
"""


def test_bounded_store(tmp_path):
    src, exe = tmp_path / "store.cpp", tmp_path / "store"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", HOST, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines()
    assert out == ["0:100 = 4", "0:100 1:101 = 8", "0:100 1:101 2:102 = 10", "1:101 2:102 3:103 = 7", "1:111 2:102 3:103 = 6",
                   "1:111 3:103 4:104 = 9", "4:104 = 5", "5:105 = 25", "6:106 = 1", "= 0", "7:107 = 10"]
