"""The panel tile's planner on the host: every product the tile's shape rule
admits has a plan, with and without workspace, and the plan covers the product;
the routes beside it. No GPU is used."""
import ctypes
import random

import pytest

import nuclis_amd as nq


def plan(encoding, rows, columns, tokens, max_floats, in_stride=None, cus=256):
    f = nq.lib().nuq_panel_plan
    u32, u64 = ctypes.c_uint32, ctypes.c_uint64
    f.argtypes = [u32, u32, u32, u32, u64, u64, u64, u32, u64 * 9]
    out = (u64 * 9)()
    ok = f(encoding, rows, columns, tokens, nq.row_bytes(encoding, columns), in_stride or columns, max_floats, cus, out)
    return list(out) if ok else None


def check(encoding, rows, columns, tokens, max_floats):
    where = f"enc {encoding} {rows}x{columns} tokens {tokens} workspace {max_floats}"
    p = plan(encoding, rows, columns, tokens, max_floats)
    assert p is not None, where
    shape, full, tail, splits, floats, bm, bn, sets, ns = p
    assert ns > 0, where
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


@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
@pytest.mark.parametrize("tokens", [65, 96, 128, 200])
def test_one_block_rows_take_tiles_of_one_group(encoding, tokens):
    """Rows of one block leave a tile nothing but its start-up: tiles of 32
    tokens (4096 x 256 at 96 tokens IQ4_XS 5.5 us, 12.7 in tiles of 128; 5.0
    and 8.1 for Q4_K)."""
    for rows in (64, 1024, 4096):
        assert plan(encoding, rows, 256, tokens, 1 << 26)[5] == 32, rows


@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
def test_few_tiles_are_split(encoding):
    """Matrices of few rows and long rows: their few tiles are split as far as
    24 ways or the blocks go, though that leaves CUs idle (64 x 17408 at 200
    tokens: IQ4_XS 16 us, 119 whole)."""
    for rows, columns, least in ((64, 17408, 16), (512, 17408, 8), (64, 5120, 10), (512, 5120, 4), (8, 4096, 8)):
        for tokens in (65, 128, 200, 512):
            p = plan(encoding, rows, columns, tokens, 1 << 26)
            assert p[1] == 0 and p[3] * p[7] >= least, (rows, columns, tokens, p)


@pytest.mark.parametrize("cus", [256, 128, 304])
def test_split_tails_leave_whole_rounds(cus):
    """Where only the tiles of a partial last round are split, the whole tiles
    fill the rounds of the CUs that are there."""
    seen = 0
    for rows in range(1024, 17409, 1024):
        for tokens in range(256, 4097, 256):
            p = plan(12, rows, 5120, tokens, 1 << 26, cus=cus)
            if p[1] and p[2]:
                seen += 1
                assert p[1] % cus == 0, (rows, tokens, p)
    assert seen


def test_refuses_what_the_tile_cannot_address():
    """Copies use 32-bit offsets within a tile; 64-column remainders and other
    encodings have no panel form."""
    assert plan(12, 64, 320, 100, 0) is None
    assert nq.lib().nuq_panel_plan(0, 64, 256, 100, 144, 256, 0, 256, (ctypes.c_uint64 * 9)()) == 0
    assert plan(12, 64, 256, 100, 0, in_stride=1 << 23) is None
    assert plan(12, 64, 256, 100, 0, in_stride=1 << 22) is not None


# encoding, rows, columns, tokens, us on the register verify tile, us on the
# panel tile: f16 activations, measured on MI355X
MEASURED = [
    (8, 4096, 9216, 4, 13.9, 18.4), (8, 4096, 9216, 16, 23.3, 19.1),
    (8, 8192, 4096, 4, 16.7, 17.8), (8, 8192, 4096, 16, 20.3, 18.6),
    (8, 4096, 14336, 4, 26.3, 22.9), (8, 4096, 14336, 16, 40.1, 23.2),
    (8, 5120, 17408, 4, 55.4, 38.3), (8, 5120, 17408, 16, 76.2, 40.0),
    (8, 17408, 5120, 4, 48.6, 38.1), (8, 17408, 5120, 16, 66.8, 40.2),
    (8, 1024, 32768, 4, 56.0, 19.2), (8, 1024, 32768, 16, 82.7, 19.9),
    (8, 16384, 2048, 4, 17.7, 15.6), (8, 16384, 2048, 16, 18.9, 16.0),
    (8, 28672, 8192, 4, 129.7, 86.5), (8, 28672, 8192, 16, 174.6, 86.9),
    (8, 7168, 7168, 4, 21.0, 22.0), (8, 7168, 7168, 16, 26.0, 22.5),
    (8, 12288, 6144, 4, 39.4, 28.6), (8, 12288, 6144, 16, 50.0, 30.3),
    (14, 4096, 9216, 4, 14.3, 19.5), (14, 4096, 9216, 16, 18.1, 17.5),
    (14, 8192, 4096, 4, 12.4, 15.5), (14, 8192, 4096, 16, 13.5, 16.2),
    (14, 4096, 14336, 4, 18.8, 21.1), (14, 4096, 14336, 16, 25.0, 21.6),
    (14, 5120, 17408, 4, 36.9, 28.2), (14, 5120, 17408, 16, 43.4, 29.1),
    (14, 17408, 5120, 4, 33.9, 27.3), (14, 17408, 5120, 16, 40.0, 28.4),
    (14, 1024, 32768, 4, 49.9, 16.8), (14, 1024, 32768, 16, 65.9, 17.4),
    (14, 16384, 2048, 4, 14.4, 12.8), (14, 16384, 2048, 16, 14.8, 13.2),
    (14, 28672, 8192, 4, 74.3, 64.7), (14, 28672, 8192, 16, 97.8, 68.0),
    (14, 7168, 7168, 4, 17.9, 19.4), (14, 7168, 7168, 16, 20.3, 20.3),
    (14, 12288, 6144, 4, 28.5, 23.6), (14, 12288, 6144, 16, 33.7, 26.3),
    (23, 4096, 9216, 4, 10.8, 18.7), (23, 4096, 9216, 16, 17.6, 16.6),
    (23, 8192, 4096, 4, 12.0, 13.7), (23, 8192, 4096, 16, 17.4, 15.0),
    (23, 4096, 14336, 4, 13.8, 20.5), (23, 4096, 14336, 16, 27.3, 21.1),
    (23, 5120, 17408, 4, 27.6, 27.6), (23, 5120, 17408, 16, 38.5, 28.6),
    (23, 17408, 5120, 4, 26.0, 27.4), (23, 17408, 5120, 16, 36.4, 29.0),
    (23, 1024, 32768, 4, 27.6, 15.1), (23, 1024, 32768, 16, 50.6, 15.8),
    (23, 16384, 2048, 4, 14.7, 11.2), (23, 16384, 2048, 16, 16.6, 11.6),
    (23, 28672, 8192, 4, 59.0, 59.8), (23, 28672, 8192, 16, 89.3, 60.4),
    (23, 7168, 7168, 4, 17.7, 19.4), (23, 7168, 7168, 16, 21.9, 20.5),
    (23, 12288, 6144, 4, 23.5, 23.5), (23, 12288, 6144, 16, 30.8, 23.8),
]
VERIFY, PANEL, PREFILL = 0, 1, 2  # TilePlan::Route


def route(encoding, rows, columns, tokens, x_f16):
    f = nq.lib().nuq_tile_route
    f.argtypes = [ctypes.c_uint32] * 5
    return f(encoding, rows, columns, tokens, x_f16)


def test_few_tokens_take_the_faster_tile():
    """4 to 16 f16 tokens on large matrices: the predicted choice is never much
    slower than the other tile."""
    for encoding, rows, columns, tokens, verify, panel in MEASURED:
        r = route(encoding, rows, columns, tokens, 1)
        assert r in (VERIFY, PANEL)
        chosen = panel if r == PANEL else verify
        assert chosen <= 1.16 * min(verify, panel), (encoding, rows, columns, tokens, r, verify, panel)


@pytest.mark.parametrize("encoding", [8, 14, 23])
def test_few_f32_tokens_and_small_matrices(encoding):
    """F32 activations take the panel tile from 4 tokens and 2^25 weights, the
    verify tile below."""
    for tokens in (4, 9, 16):
        assert route(encoding, 4096, 8192, tokens, 0) == PANEL
        assert route(encoding, 4088, 8192, tokens, 0) == route(encoding, 4088, 8192, tokens, 1) == VERIFY
    assert route(encoding, 1 << 15, 1 << 15, 3, 0) == route(encoding, 1 << 15, 1 << 15, 3, 1) == VERIFY
    for e in (12, 13):
        assert route(e, 5120, 17408, 16, 0) == route(e, 5120, 17408, 48, 1) == VERIFY
        assert route(e, 5120, 17408, 49, 0) == route(e, 5120, 17408, 49, 1) == PANEL


# rows, columns, tokens, us on the prefill tile, us on the panel tile: Q8_0 with
# f16 activations on matrices of few rows or short rows, measured on MI355X
MEASURED_Q8 = [
    (64, 17408, 64, 37.7, 14.0), (64, 17408, 200, 37.6, 16.8), (64, 17408, 512, 41.7, 18.6),
    (64, 17408, 1024, 42.8, 21.0), (512, 5120, 64, 23.2, 11.8), (512, 5120, 200, 23.7, 15.7),
    (512, 5120, 512, 26.5, 20.6), (512, 5120, 1024, 26.9, 22.7), (4096, 256, 64, 12.1, 6.7),
    (4096, 256, 200, 13.5, 7.2), (4096, 256, 512, 14.8, 11.0), (4096, 256, 1024, 16.2, 13.3),
    (17408, 256, 64, 12.9, 10.1), (17408, 256, 512, 17.4, 25.7), (17408, 512, 64, 19.2, 11.6),
    (17408, 512, 512, 24.7, 31.5), (17408, 1280, 64, 36.1, 20.4), (17408, 1280, 512, 41.5, 50.0),
    (17408, 1280, 1024, 67.5, 83.1), (8192, 2048, 64, 31.9, 16.0), (8192, 2048, 200, 32.6, 21.9),
    (8192, 2048, 512, 46.1, 33.8), (8192, 2048, 1024, 60.8, 53.8),
]


def test_q8_takes_the_faster_tile():
    """Short rows leave the results' stores, long rows of few tiles the split:
    Q8_0 runs on the tile that is the faster one there."""
    for rows, columns, tokens, prefill, panel in MEASURED_Q8:
        r = route(8, rows, columns, tokens, 1)
        assert r in (PANEL, PREFILL)
        chosen = panel if r == PANEL else prefill
        assert chosen <= 1.1 * min(prefill, panel), (rows, columns, tokens, r, prefill, panel)
