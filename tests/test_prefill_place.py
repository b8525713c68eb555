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
// Batches of up to `rows` queries within `capacity` positions that need more
// workspace than the bounds (p0 and the length in steps of their own).
extern "C" int exceeding(int rows, int heads, int kv_heads, int capacity)
{
    int bad = 0;
    for (int n = 1; n <= rows && n <= capacity; n += n < 70 ? 1 : 13)
        for (int p0 = capacity - n, i = 0; p0 >= 0 && i < 70; p0 -= i < 40 ? 1 : 101, ++i) {
            const PaBatch b{p0, n, kv_heads, heads / kv_heads};
            bad += pa_takes_partials(b) ? pa_partials(b) > pa_max_partials(rows, heads, capacity)
                                        : pa_tile_chunks(b) > pa_max_tile_chunks(rows, capacity);
        }
    return bad;
}
"""


@pytest.fixture(scope="module")
def place(tmp_path_factory):
    d = tmp_path_factory.mktemp("place")
    (d / "place.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", f"-I{CSRC}", str(d / "place.cpp"), "-o",
                    str(d / "place.so")], check=True)
    return ctypes.CDLL(str(d / "place.so"))


@pytest.mark.parametrize("kv_heads,groups", [(8, 4), (8, 2), (8, 1), (2, 3), (4, 8), (2, 5), (1, 1), (3, 7)])
def test_every_output_and_partial_has_one_writer(place, kv_heads, groups):
    # starts inside and on the edges of a query tile and of a chunk; lengths
    # that end in the first chunk, just past it and several chunks on
    for p0 in (0, 1, 15, 16, 17, 20, 31, 32, 33, 47, 48, 60, 63, 64, 65, 100, 127, 128, 1000):
        for rows in (1, 2, 15, 16, 17, 33, 45, 48, 64, 66, 130, 300):
            for part in (0, 1):
                assert place.misplaced(p0, rows, kv_heads, groups, part) == 0, (p0, rows, part)


def test_whole_passes_have_one_writer_each(place):
    # launches of several rounds of blocks (the second round's order is turned)
    for p0, rows, kv_heads, groups in ((0, 2048, 8, 4), (5, 2000, 8, 2), (2048, 1100, 2, 3), (7, 1024, 1, 8)):
        assert place.misplaced(p0, rows, kv_heads, groups, 0) == 0, (p0, rows, kv_heads, groups)


@pytest.mark.parametrize("heads,kv_heads", [(32, 8), (16, 8), (3, 3), (6, 2), (64, 8), (1, 1), (40, 8)])
def test_workspace_bounds_hold_every_batch(place, heads, kv_heads):
    for capacity in (1, 15, 16, 17, 63, 64, 65, 500, 513, 2047, 2048, 2063, 2064, 2065, 3000, 4111, 9001):
        assert place.exceeding(min(2048, capacity), heads, kv_heads, capacity) == 0, capacity


def _model(**changes):
    from harsh4b_amd import _native
    m = _native.HqModel()
    shape = dict(layers=36, hidden=2560, intermediate=9728, heads=32, kv_heads=8, head_dim=128, vocab=151936,
                 rope_positions=40960, **changes)
    for name, value in shape.items():
        setattr(m, name, value)
    m.layer = (_native.HqLayer * 1)()      # (only its presence is looked at)
    return m


def test_prefill_workspace_bytes():
    # the 4B shape: the activations of 2048 tokens and the scores or partials
    # of the batches a cache can hold, never less for a larger cache (a call
    # uses the layout of its own last position)
    from harsh4b_amd import _native
    lib, m = _native.lib(), _model()
    size = {c: lib.hq_prefill_workspace_bytes(ctypes.byref(m), c)
            for c in [*range(1, 300), *range(2000, 2200), 4096, 8192, 40960]}
    sizes = [size[c] for c in sorted(size)]
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))
    assert size[64] < 20 << 20
    assert size[2048] < 480 << 20
    assert size[4096] < 1024 << 20
    assert size[40960] < 1232 << 20
