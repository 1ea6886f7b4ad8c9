"""Which head and tile a workgroup of a backward launch takes (non-causal), on the library's own index arithmetic compiled for the host:
every tile exactly once, and a head's tiles on as few of the 8 compute dies as the order promises -- one for a dealt head, a range of
neighbouring workgroups for the others wherever their number divides by 8 (heads left over behind groups of eight, launches of fewer
than eight heads and of full mask tensors among them)."""
import os
import subprocess

import pytest

from nvfuserexamples_amd import build as B

PROGRAM = r"""
#include "fmha_bwd_kernel.h"
#include <cstdio>
int main() {
  int kind, bh, units, others;
  while (std::scanf("%d %d %d %d", &kind, &bh, &units, &others) == 4) {
    const int dealt = kind >= 0 && fmha::bwd_heads_dealt(kind != 0, bh, units, others) ? fmha::bwd_dealt_blocks(bh, units) : 0, nb = bh * units;
    std::printf("%d", dealt);
    for (int bid = 0; bid < nb; ++bid) {
      int head, unit;
      fmha::bwd_head_and_unit(bid, dealt, fmha::bwd_range_blocks(nb, dealt), units, head, unit);
      std::printf(" %d", head * units + unit);
    }
    std::printf("\n");
  }
  const int64_t rows[][3] = {{1, 0, 80}, {16, 80, 3840}, {16, 64, 3072}, {16, 128, 6144}, {8, 96, 2304}, {8, 40960, 80}, {8, 0, 64}};
  for (const auto &r : rows) std::printf("%d ", (int)fmha::rows_share_lines((int)r[0], r[1], r[2]));
}
"""
NOT, WHOLE, SHARED = -1, 0, 1  # no lengths that may differ; rows in cache lines of their own; lines shared by neighbouring heads
LAUNCHES = [(kind, bh, units, others) for kind in (NOT, WHOLE, SHARED) for bh in (1, 4, 7, 8, 9, 12, 20, 36, 60, 64, 272)
            for units in (1, 2, 3, 4, 5, 7, 8, 16, 32) for others in (1, 4, 9)]


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_heads_of_a_backward_launch_on_the_compute_dies(tmp_path):
    src, exe = tmp_path / "order.cpp", str(tmp_path / "order")
    src.write_text(PROGRAM)
    subprocess.run([B.HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-I", B.CSRC, str(src), "-o", exe], check=True,
                   capture_output=True)
    text = "\n".join("%d %d %d %d" % x for x in LAUNCHES)
    out = subprocess.run([exe], input=text, check=True, capture_output=True, text=True).stdout.split("\n")
    for (kind, bh, units, others), line in zip(LAUNCHES, out):
        dealt, *item = map(int, line.split())
        nb, name = bh * units, (kind, bh, units, others)
        assert sorted(item) == list(range(nb)), name
        ranges = nb % 8 == 0 and bh * others % 8 == 0  # to be had, for dQ and for dK / dV
        wanted = kind != NOT and max(units, others) >= (2 if not ranges else 5 if kind == SHARED else 3)
        assert dealt == (bh // 8 * 8 * units if wanted else 0), name
        dies = [{i & 7 for i in range(nb) if item[i] // units == head} for head in range(bh)]
        assert all(len(d) == 1 for d in dies[:dealt // units]), name
        if (nb - dealt) % 8 == 0 and nb > dealt:
            per_die = (nb - dealt) // 8  # neighbouring tiles of one die
            assert all(len(d) <= (units - 1 + per_die - 1) // per_die + 1 for d in dies[dealt // units:]), name
    assert out[len(LAUNCHES)].split() == list("0100101")
