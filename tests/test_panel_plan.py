"""The panel tile's planner on the host: every product the tile's shape rule
admits has a plan, with and without workspace, and the plan covers the product.
No GPU is used (the cost model then assumes 256 compute units)."""
import ctypes
import random

import pytest

import nuclis_amd as nq


def plan(encoding, rows, columns, tokens, max_floats, in_stride=None):
    f = nq.lib().nuq_panel_plan
    u32, u64 = ctypes.c_uint32, ctypes.c_uint64
    f.argtypes = [u32, u32, u32, u32, u64, u64, u64, u64 * 8]
    out = (u64 * 8)()
    ok = f(encoding, rows, columns, tokens, nq.row_bytes(encoding, columns), in_stride or columns, max_floats, out)
    return list(out) if ok else None


def check(encoding, rows, columns, tokens, max_floats):
    where = f"enc {encoding} {rows}x{columns} tokens {tokens} workspace {max_floats}"
    p = plan(encoding, rows, columns, tokens, max_floats)
    assert p is not None, where
    shape, full, tail, splits, floats, bm, bn, sets = p
    nb = columns // 256
    assert full + tail == -(-tokens // bm) * -(-rows // bn), where
    # every wave set of every split has a 256-column block
    assert splits * sets <= nb and (splits == 1) == (tail == 0), where
    assert floats == tail * splits * bm * bn * (splits > 1) <= max_floats, where


@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
def test_every_product_has_a_plan(encoding):
    """Blocks per row from one (no second K set) and every token count over
    several rounds of token groups, then random shapes."""
    for nb in (1, 2, 3, 4):
        for tokens in range(1, 301):
            for rows, floats in ((8, 0), (8, 1 << 26), (5120, 1 << 26)):
                check(encoding, rows, 256 * nb, tokens, floats)
    rng = random.Random(5)
    for _ in range(2000):
        check(encoding, 8 * rng.randint(1, 4000), 256 * rng.randint(1, 80), int(2 ** rng.uniform(0, 13)),
              rng.choice([0, 1 << 20, 1 << 26]))


def test_refuses_what_the_tile_cannot_address():
    """Copies use 32-bit offsets within a tile; 64-column remainders and other
    encodings have no panel form."""
    assert plan(12, 64, 320, 100, 0) is None
    assert nq.lib().nuq_panel_plan(0, 64, 256, 100, 144, 256, 0, (ctypes.c_uint64 * 8)()) == 0
    assert plan(12, 64, 256, 100, 0, in_stride=1 << 23) is None
    assert plan(12, 64, 256, 100, 0, in_stride=1 << 22) is not None
