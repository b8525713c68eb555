"""Placement of the prompt attention's blocks and waves, from the kernels' own
header compiled for the host: every output and every chunk partial has exactly
one writer."""
import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "harsh4b_amd" / "csrc"

# The kernels' loops (hq_prefill_attn.hip) over a whole grid, counting writers.
# out [rows][heads]: by the waves themselves; a query of several chunks gets
# its output from the combine when the launch writes partials.  Returns the
# number of entries that do not have exactly the writers they should.
SOURCE = r"""
#include <stddef.h>
#include <vector>
#include "hq_prefill_place.h"
using namespace hq;
extern "C" int misplaced(int p0, int rows, int kv_heads, int groups, int part)
{
    const PaBatch b{p0, rows, kv_heads, groups};
    const int heads = kv_heads * groups, nc_max = (p0 + rows - 1) / kPaChunk + 1;
    const size_t n = size_t(rows) * heads;
    std::vector<int> out(n), partial(n * nc_max);
    const PaPartGrid g = part ? pa_part_grid(b) : PaPartGrid{pa_blocks_per_kv(b) * kv_heads, 1, nc_max};
    for (int x = 0; x < g.blocks; ++x)
        for (int y = 0; y < g.splits; ++y)
            for (int wave = 0; wave < kPaWaves; ++wave) {
                const PaSlot s = pa_slot(b, x, wave);
                const int c_begin = y * g.cpb, c_end = pa_min(s.nc_block, c_begin + g.cpb);
                if (c_begin >= c_end || !s.live) continue;
                for (int i = 0; i < kPaTile; ++i) {
                    const int pos = s.tile * kPaTile + i, z = pos - p0;
                    if (z < 0 || z >= rows) continue;
                    for (int c = c_begin; c < c_end && c < s.nc; ++c)
                        if (part && s.nc > 1) ++partial[(size_t(z) * heads + s.h) * nc_max + c];
                    if (pa_stores_output(part != 0, s.nc, c_begin)) ++out[size_t(z) * heads + s.h];
                }
            }
    int bad = 0;
    for (int z = 0; z < rows; ++z)
        for (int h = 0; h < heads; ++h) {
            const int nc = (p0 + z) / kPaChunk + 1;
            bad += out[size_t(z) * heads + h] != (part && nc > 1 ? 0 : 1);
            for (int c = 0; c < nc_max; ++c)
                bad += partial[(size_t(z) * heads + h) * nc_max + c] != (part && nc > 1 && c < nc ? 1 : 0);
        }
    return bad;
}
"""


@pytest.fixture(scope="module")
def misplaced(tmp_path_factory):
    d = tmp_path_factory.mktemp("place")
    (d / "place.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", f"-I{CSRC}", str(d / "place.cpp"), "-o",
                    str(d / "place.so")], check=True)
    return ctypes.CDLL(str(d / "place.so")).misplaced


@pytest.mark.parametrize("kv_heads,groups", [(8, 4), (8, 2), (8, 1), (2, 3), (4, 8), (2, 5), (1, 1), (3, 7)])
def test_every_output_and_partial_has_one_writer(misplaced, kv_heads, groups):
    # starts inside and on the edges of a query tile and of a chunk; lengths
    # that end in the first chunk, just past it and several chunks on
    for p0 in (0, 1, 15, 16, 17, 20, 31, 32, 33, 47, 48, 60, 63, 64, 65, 100, 127, 128, 1000):
        for rows in (1, 2, 15, 16, 17, 33, 45, 48, 64, 66, 130, 300):
            for part in (0, 1):
                assert misplaced(p0, rows, kv_heads, groups, part) == 0, (p0, rows, part)


def test_whole_passes_have_one_writer_each(misplaced):
    # launches of several rounds of blocks (the second round's order is turned)
    for p0, rows, kv_heads, groups in ((0, 2048, 8, 4), (5, 2000, 8, 2), (2048, 1100, 2, 3), (7, 1024, 1, 8)):
        assert misplaced(p0, rows, kv_heads, groups, 0) == 0, (p0, rows, kv_heads, groups)
