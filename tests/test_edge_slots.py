"""Bounds of the positions that the sparse kernels' lanes read, on the host: every lane of a row loads, also past the row's end
and in rows without edges, so every position it names has to be one of the graph's edges."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torchgt_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include "edge_slots.h"
int main() {
    int start, n, slot;
    while (std::scanf("%d %d %d", &start, &n, &slot) == 3) std::printf("%d\n", tgt::edge_of_slot(start, n, slot));
}
"""


def test_positions_stay_inside_the_edge_list(tmp_path):
    src, exe = tmp_path / "slots.cpp", tmp_path / "slots"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-D__host__=", "-D__device__=", "-D__forceinline__=inline", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    asked = []      # (start, n, slot, E)
    for degrees in ([0, 3, 0, 1, 0, 0], [5], [0, 1], [2, 0], [33, 0, 16, 0]):
        E, start = sum(degrees), 0
        for n in degrees:
            asked += [(start, n, slot, E) for slot in range(64)]
            start += n
    out = subprocess.run([str(exe)], input="".join(f"{a} {b} {c}\n" for a, b, c, _ in asked), capture_output=True, text=True, check=True).stdout.split()
    assert len(out) == len(asked)
    for (start, n, slot, E), got in zip(asked, map(int, out)):
        assert 0 <= got < E, f"row at {start} with {n} of {E} edges, slot {slot}: position {got}"
        if n > 0:
            assert got == start + min(slot, n - 1)
