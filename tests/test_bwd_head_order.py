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
  int kind, bh, units;
  while (std::scanf("%d %d %d", &kind, &bh, &units) == 3) {
    const int dealt = kind < 0 ? 0 : fmha::bwd_dealt_blocks(kind == 2, kind == 1, bh, units), nb = bh * units;
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
NO_MASK, WHOLE, SHARED, ONE = -1, 0, 1, 2  # no lengths that may differ; rows in cache lines of their own; lines shared by neighbouring
# heads; many heads of one tile at head dim 256
LAUNCHES = [(kind, bh, units) for kind in (NO_MASK, WHOLE, SHARED, ONE) for bh in (1, 4, 7, 8, 9, 12, 20, 36, 60, 64, 272)
            for units in (1, 2, 3, 4, 5, 7, 8, 16, 32)]


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_heads_of_a_backward_launch_on_the_compute_dies(tmp_path):
    src, exe = tmp_path / "order.cpp", str(tmp_path / "order")
    src.write_text(PROGRAM)
    subprocess.run([B.HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-I", B.CSRC, str(src), "-o", exe], check=True,
                   capture_output=True)
    text = "\n".join("%d %d %d" % x for x in LAUNCHES)
    out = subprocess.run([exe], input=text, check=True, capture_output=True, text=True).stdout.split("\n")
    for (kind, bh, units), line in zip(LAUNCHES, out):
        dealt, *item = map(int, line.split())
        nb, name = bh * units, (kind, bh, units)
        assert sorted(item) == list(range(nb)), name
        wanted = kind != NO_MASK and (units >= (2 if nb % 8 else 8 if kind == SHARED else 3) or (kind == ONE and units == 1))
        assert dealt == (bh // 8 * 8 * units if wanted else 0), name
        dies = [{i & 7 for i in range(nb) if item[i] // units == head} for head in range(bh)]
        assert all(len(d) == 1 for d in dies[:dealt // units]), name
        if (nb - dealt) % 8 == 0 and nb > dealt:
            per_die = (nb - dealt) // 8  # neighbouring tiles of one die
            assert all(len(d) <= (units - 1 + per_die - 1) // per_die + 1 for d in dies[dealt // units:]), name
    assert out[len(LAUNCHES)].split() == list("0100101")
