"""Every shape of the panel tile, in every encoding, against the CPU oracle:
ragged rows and tokens (a last tile of one row group and of one token past a
32-token group), K ranges of unequal length among the wave sets, whole tiles,
all tiles split along K and a split tail. The plan is forced, so each shape runs at a small size; the routed
entry is then checked for the f16 copy of F32 activations and for capture."""
import ctypes

import numpy as np
import pytest

import nuclis_amd as nq
from nuclis_amd.synth import gaussian
from oracle import oracle as orc
from tests.gpu_util import F16_K, check_close, mass, to_gpu

pytestmark = pytest.mark.gpu

# TG, RG, WR, WK, DEPTH of the library's shapes (test_shape_table)
SHAPES = [(1, 1, 4, 1, 4), (1, 1, 2, 4, 2), (2, 1, 2, 2, 2), (3, 1, 4, 2, 2), (4, 1, 4, 2, 2),
          (4, 1, 2, 2, 2), (4, 1, 4, 1, 2), (4, 2, 4, 1, 2), (6, 2, 4, 1, 2), (8, 2, 4, 1, 2)]


@pytest.fixture(scope="module")
def backend():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    b = nq.Backend(0)
    yield b
    b.close()


def launch(encoding, w, x, columns, y, shape, full, tail, splits, work):
    """One product on the given plan: w [rows][bytes], x [tokens][stride], y
    [tokens][stride], all on the GPU; rows come with `w`, tokens with `x`."""
    import torch
    f, u32, u64, vp = nq.lib().nuq_panel_run, ctypes.c_uint32, ctypes.c_uint64, ctypes.c_void_p
    f.argtypes = [vp, u32, vp, u64, u32, u32, vp, u64, vp, u64, u32, u32, u32, u32, u32, vp]
    return f(torch.cuda.current_stream().cuda_stream, encoding, w.data_ptr(), w.shape[1], w.shape[0], columns,
             x.data_ptr(), x.shape[1], y.data_ptr(), y.shape[1], x.shape[0], shape, full, tail, splits, work.data_ptr())


def test_shape_table(backend):
    out = (ctypes.c_uint32 * 5)()
    table = []
    while nq.lib().nuq_panel_shape(len(table), out):
        table.append(tuple(out))
    assert table == SHAPES


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
def test_every_shape_matches_oracle(backend, encoding, shape):
    import torch
    tg, rg, wr, wk, _ = SHAPES[shape]
    bm, bn = 32 * tg, 32 * rg * wr
    rows, tokens, columns = bn + 40, bm + 33, 256 * (2 * wk + 1)
    in_stride, out_stride = columns + 8, rows + 3
    print(f"[panel] enc {encoding} shape {shape} {rows}x{columns} tokens {tokens}", flush=True)
    w = nq.quantize(encoding, gaussian(31 + shape, (rows, columns), 0.02))
    x = gaussian(7 + encoding, (tokens, in_stride)).astype(np.float16)
    wg, xg = to_gpu(w), to_gpu(x)
    check = sorted({0, 1, 31, 32, bm - 1, bm, bm + 31, bm + 32} & set(range(tokens)))
    xr = x[check, :columns].astype(np.float32)
    want, m = orc.matmul(encoding, rows, columns, w, xr), mass(encoding, w, rows, columns, xr)
    tiles = -(-tokens // bm) * -(-rows // bn)
    work = torch.empty(tiles * 2 * bm * bn, device="cuda")
    for full, tail, splits in ((tiles, 0, 1), (0, tiles, 2), (tiles - 1, 1, 2)):
        y = torch.full((tokens, out_stride), np.nan, device="cuda")
        assert launch(encoding, wg, xg, columns, y, shape, full, tail, splits, work) == 0
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert np.isnan(got[:, rows:]).all() and np.isfinite(got[:, :rows]).all()
        check_close(got[check, :rows], want, m, F16_K, f"panel {encoding} shape {shape} splits {splits} tail {tail}")


def run_shape(encoding, shape, w, x, splits=1):
    """The product on one forced shape: [tokens][rows]."""
    import torch
    tg, rg, wr, wk, _ = SHAPES[shape]
    bm, bn = 32 * tg, 32 * rg * wr
    rows, tokens, columns = w.shape[0], *x.shape
    tiles = -(-tokens // bm) * -(-rows // bn)
    wg, xg, y = to_gpu(w), to_gpu(x), torch.full((tokens, rows), float("nan"), device="cuda")
    work = torch.empty(tiles * splits * bm * bn, device="cuda")
    assert launch(encoding, wg, xg, columns, y, shape, tiles if splits == 1 else 0, 0 if splits == 1 else tiles, splits,
                  work) == 0
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
def test_weights_are_the_decoded_values_in_f16(backend, encoding, shape):
    """Every weight is the CPU decoder's F32 value rounded to f16 and nothing
    else, so against those weights in float64 only the F32 sums are left:
    activations of a non-zero mean show an offset that a group shares."""
    wk = SHAPES[shape][3]
    rows, tokens, columns = 200, 40, 256 * max(2, wk)
    print(f"[panel-exact] enc {encoding} shape {shape}", flush=True)
    w = nq.quantize(encoding, gaussian(61 + shape, (rows, columns), 0.02))
    x = (gaussian(62, (tokens, columns)) + 1).astype(np.float16)
    dec = orc.decode_matrix(encoding, w, rows, columns).astype(np.float16).astype(np.float64)
    got = run_shape(encoding, shape, w, x)
    want, m = x.astype(np.float64) @ dec.T, np.abs(x.astype(np.float64)) @ np.abs(dec).T
    # at most columns / 16 + 4 F32 roundings of a running sum (16 products of
    # the matrix core's inner sum, the K sets and halves), each of at most
    # 2^-24 of the mass; the core's own alignment of 16 products adds as much
    bound = 2 * (columns / 16 + 4) * 2.0**-24 * m
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / m).max())


def blocks(encoding, rows, columns, seed):
    """Random blocks with ordinary scales: [rows][blocks][block bytes]."""
    values, size = nq.LAYOUT[encoding]
    return nq.quantize(encoding, gaussian(seed, (rows, columns), 0.02)).reshape(rows, columns // values, size).copy()


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("encoding", [12, 13])
def test_zero_weights_meet_infinity(backend, encoding, shape):
    """A weight of exactly zero (d sc q = dmin m) times an infinite activation
    is NaN, as in the CPU reference; all other rows give an infinity."""
    rows, tokens, columns = 200, 40, 256 * max(2, SHAPES[shape][3])
    b = blocks(encoding, rows, columns, 71)
    b[..., 2:4] = b[..., 0:2] = np.random.default_rng(72).integers(0x1800, 0x2400, b.shape[:2], dtype=np.uint16)[..., None].view(np.uint8)
    w = b.reshape(rows, -1)
    dec = orc.decode_matrix(encoding, w, rows, columns)
    x = np.ones((tokens, columns), np.float16)
    cols = np.argsort(-(dec == 0).sum(0))[:tokens]  # the columns with most zeros
    x[np.arange(tokens), cols] = np.inf
    want_nan = (dec[:, cols] == 0).T
    assert want_nan.any() and not want_nan.all()
    got = run_shape(encoding, shape, w, x)
    assert np.array_equal(np.isnan(got), want_nan)
    assert np.array_equal(np.isposinf(got), (dec[:, cols] > 0).T) and np.array_equal(np.isneginf(got), (dec[:, cols] < 0).T)


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
def test_infinite_scales_keep_the_weights_signs(backend, encoding, shape):
    """A block of infinite scale: +-Inf for codes of one sign, NaN for a zero
    code (rows 1 mod 4) and for a scale of zero (rows 2 mod 4); rows 0 mod 4
    are finite."""
    rows, tokens, columns = 200, 40, 512 * SHAPES[shape][3]
    values, _ = nq.LAYOUT[encoding]
    b = blocks(encoding, rows, columns, 81)
    sick = np.arange(rows) % 4 != 0
    at = (columns // values) - 1  # in the last block, also a unit's second half for Q8_0
    d = {8: 0, 12: 0, 13: 0, 14: 208, 23: 0}[encoding]
    sign = np.where(np.arange(rows) % 8 == 3, 0x7c00, 0xfc00).astype(np.uint16)
    blk = b[:, at]
    if encoding == 8:
        blk[:, 2:] = 5
        blk[1::4, 9] = 0
        blk[2::4, 2:] = 0
    elif encoding in (12, 13):
        blk[:, 2:4] = 0                       # dmin = 0
        blk[:, 4:16] = 0x2f
        blk[:, -128:] |= 0x11                 # no zero code
        blk[1::4, -128 + 37] = 0
        if encoding == 13:
            blk[1::4, 16:48] = 0
        blk[2::4, 4:16] = 0
    elif encoding == 14:
        blk[:, :128], blk[:, 128:192], blk[:, 192:208] = 0x55, 0xaa, 3   # codes 37
        blk[1::4, 77] = 0x50                  # one code of 32
        blk[2::4, 199] = 0
    else:
        blk[:, 2:4], blk[:, 4:8] = 0xff, 0x11
        blk[:, 8:] |= 0x88                    # positive values
        blk[2::4, 2:4], blk[2::4, 4:8] = 0xaa, 0x00  # scales of zero
    blk[sick, d:d + 2] = sign[sick].view(np.uint8).reshape(-1, 2)
    w = b.reshape(rows, -1)
    dec = orc.decode_matrix(encoding, w, rows, columns).astype(np.float64)
    x = np.abs(gaussian(82, (tokens, columns))).astype(np.float16) + np.float16(0.5)
    with np.errstate(invalid="ignore"):
        want = (dec[None] * x.astype(np.float64)[:, None, :]).sum(-1)
    assert np.isposinf(want).any() and np.isneginf(want).any() and np.isnan(want).any()
    assert np.isfinite(want[:, ~sick]).all()
    for splits in (1, 2):
        got = run_shape(encoding, shape, w, x, splits)
        for cls in (np.isnan, np.isposinf, np.isneginf):
            assert np.array_equal(cls(got), cls(want)), (cls.__name__, splits)


@pytest.mark.parametrize("splits", [2, 4, 5, 6, 9, 11])
def test_partial_sums_of_any_split_count(backend, splits):
    """The reduction reads four splits at a time: counts around its turns."""
    import torch
    rows, tokens, columns = 136, 33, 256 * 11
    w = nq.quantize(14, gaussian(41, (rows, columns), 0.02))
    x = gaussian(42, (tokens, columns)).astype(np.float16)
    wg, xg = to_gpu(w), to_gpu(x)
    work, y = torch.empty(4 * splits * 32 * 128, device="cuda"), torch.full((tokens, rows), np.nan, device="cuda")
    assert launch(14, wg, xg, columns, y, 0, 0, 4, splits, work) == 0
    torch.cuda.synchronize()
    xr = x.astype(np.float32)
    check_close(y.cpu().numpy(), orc.matmul(14, rows, columns, w, xr), mass(14, w, rows, columns, xr), F16_K,
                f"panel {splits} splits")


@pytest.mark.parametrize("encoding,rows,columns,tokens", [(12, 1032, 512, 77), (14, 520, 2304, 300), (8, 4104, 2048, 260),
                                                          (8, 264, 320, 40), (23, 1024, 32768, 8)])
def test_f32_activations_equal_their_f16_rounding(backend, encoding, rows, columns, tokens):
    """The tiles round F32 activations to f16: the same bits as f16 input (where
    both kinds take the same tile)."""
    import torch
    w = to_gpu(nq.quantize(encoding, gaussian(3, (rows, columns), 0.02)))
    m = nq.Matrix(encoding, rows, columns, w)
    x = torch.randn((tokens, columns + 16), generator=torch.Generator().manual_seed(5)).cuda()
    y32, y16 = torch.empty((tokens, rows), device="cuda"), torch.empty((tokens, rows), device="cuda")
    backend.matmul(m, x, columns + 16, y32, rows, tokens)
    backend.matmul(m, x.half(), columns + 16, y16, rows, tokens)
    backend.sync()
    assert torch.equal(y32, y16)


def test_captured_f32_product_replays():
    """A captured F32 product (copy, split tiles and their reduction in the
    reserved workspace) replays to the eager bits; one captured with no
    workspace at all takes the routes that need none."""
    import torch
    rows, columns, tokens = 1544, 2560, 200
    w = nq.quantize(14, gaussian(9, (rows, columns), 0.02))
    m = nq.Matrix(14, rows, columns, to_gpu(w))
    x = torch.randn((tokens, columns), generator=torch.Generator().manual_seed(6)).cuda()
    xr = x[:4].half().float().cpu().numpy()
    want, ms = orc.matmul(14, rows, columns, w, xr), mass(14, w, rows, columns, xr)
    for reserve in (64 << 20, 0):
        b = nq.Backend(0)
        eager, y = torch.empty((tokens, rows), device="cuda"), torch.empty((tokens, rows), device="cuda")
        if reserve:
            b.reserve_workspace(reserve)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            b.matmul(m, x, columns, y, rows, tokens)
        b2 = nq.Backend(0)
        b2.matmul(m, x, columns, eager, rows, tokens)
        b2.sync()
        for _ in range(3):
            y.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            check_close(y[:4].cpu().numpy(), want, ms, F16_K, "panel-captured")
            if reserve:
                assert torch.equal(y, eager)
            assert torch.isfinite(y).all()
        b.close()
        b2.close()


@pytest.mark.parametrize("encoding,tokens", [(14, 1025), (8, 2051)])
def test_f32_activations_beyond_one_copy(backend, encoding, tokens):
    """256 MiB of f16 rows at a time: 1024 rows of 131072 columns, then a
    short last part."""
    import torch
    rows, columns = 72, 131072
    print(f"[panel] enc {encoding} {rows}x{columns} tokens {tokens} in parts", flush=True)
    w = nq.quantize(encoding, gaussian(12, (rows, columns), 0.02))
    m = nq.Matrix(encoding, rows, columns, to_gpu(w))
    x = torch.randn((tokens, columns), device="cuda", generator=torch.Generator("cuda").manual_seed(8))
    y = torch.full((tokens, rows), float("nan"), device="cuda")
    backend.matmul(m, x, columns, y, rows, tokens)
    backend.sync()
    check = [0, 1023, 1024, tokens - 1]
    xr = x[check].half().float().cpu().numpy()
    assert torch.isfinite(y).all()
    check_close(y[check].cpu().numpy(), orc.matmul(encoding, rows, columns, w, xr), mass(encoding, w, rows, columns, xr),
                F16_K, f"panel {encoding} in parts")


@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
@pytest.mark.parametrize("tokens", [65, 77, 96])
def test_one_block_rows(backend, encoding, tokens):
    """Rows of one 256-column block at 65 to 96 tokens: three token groups and
    no second K set."""
    import torch
    rows, columns = 136, 256
    w = nq.quantize(encoding, gaussian(51, (rows, columns), 0.02))
    m = nq.Matrix(encoding, rows, columns, to_gpu(w))
    x = to_gpu(gaussian(52, (tokens, columns)))
    xr = x.half().float().cpu().numpy()
    want, ms = orc.matmul(encoding, rows, columns, w, xr), mass(encoding, w, rows, columns, xr)
    for xg in (x, x.half()):
        y = torch.full((tokens, rows), float("nan"), device="cuda")
        backend.matmul(m, xg, columns, y, rows, tokens)
        backend.sync()
        check_close(y.cpu().numpy(), want, ms, F16_K, f"panel-one-block {encoding} tokens {tokens}")


@pytest.mark.parametrize("encoding", [8, 14])
def test_one_block_rows_in_parts(backend, encoding):
    """524288 tokens of 256 columns fill one f16 copy; 77 more are a last part
    of their own."""
    import torch
    rows, columns, tokens = 8, 256, 524288 + 77
    print(f"[panel] enc {encoding} {rows}x{columns} tokens {tokens} in parts", flush=True)
    w = nq.quantize(encoding, gaussian(53, (rows, columns), 0.02))
    m = nq.Matrix(encoding, rows, columns, to_gpu(w))
    x = torch.randn((tokens, columns), device="cuda", generator=torch.Generator("cuda").manual_seed(9))
    y = torch.full((tokens, rows), float("nan"), device="cuda")
    backend.matmul(m, x, columns, y, rows, tokens)
    backend.sync()
    assert torch.isfinite(y).all()
    check = [0, 524287, 524288, tokens - 1]
    xr = x[check].half().float().cpu().numpy()
    check_close(y[check].cpu().numpy(), orc.matmul(encoding, rows, columns, w, xr), mass(encoding, w, rows, columns, xr),
                F16_K, f"panel-one-block {encoding} in parts")


@pytest.mark.parametrize("encoding", [8, 14, 23])
@pytest.mark.parametrize("tokens", [4, 7, 16])
def test_few_tokens_on_a_large_matrix(backend, encoding, tokens):
    """4 to 16 tokens on 2^25 weights and more run on the panel tile."""
    import torch
    rows, columns = 8 * 129, 32768
    print(f"[panel] enc {encoding} {rows}x{columns} tokens {tokens}", flush=True)
    part = nq.quantize(encoding, gaussian(91, (129, columns), 0.02))
    m = nq.Matrix(encoding, rows, columns, to_gpu(np.tile(part, (8, 1))))
    x = to_gpu(gaussian(92, (tokens, columns)))
    xr = x.half().float().cpu().numpy()
    want, ms = (np.tile(a, 8) for a in (orc.matmul(encoding, 129, columns, part, xr), mass(encoding, part, 129, columns, xr)))
    for xg in (x, x.half()):
        y = torch.full((tokens, rows), float("nan"), device="cuda")
        backend.matmul(m, xg, columns, y, rows, tokens)
        backend.sync()
        check_close(y.cpu().numpy(), want, ms, F16_K, f"panel-few {encoding} tokens {tokens}")


@pytest.mark.parametrize("encoding", [8, 12, 13, 14, 23])
@pytest.mark.parametrize("rows,columns,tokens", [(8, 17408, 65), (64, 5120, 200), (136, 2304, 130)])
def test_few_tiles_on_long_rows(backend, encoding, rows, columns, tokens):
    """Few tiles, split as far as 24 ways or their blocks go (one or two a range)."""
    import torch
    print(f"[panel] enc {encoding} {rows}x{columns} tokens {tokens}", flush=True)
    w = nq.quantize(encoding, gaussian(95, (rows, columns), 0.02))
    m = nq.Matrix(encoding, rows, columns, to_gpu(w))
    x = to_gpu(gaussian(96, (tokens, columns)))
    xr = x.half().float().cpu().numpy()
    want, ms = orc.matmul(encoding, rows, columns, w, xr), mass(encoding, w, rows, columns, xr)
    for xg in (x, x.half()):
        y = torch.full((tokens, rows), float("nan"), device="cuda")
        backend.matmul(m, xg, columns, y, rows, tokens)
        backend.sync()
        check_close(y.cpu().numpy(), want, ms, F16_K, f"panel-few-tiles {encoding} {rows}x{columns}")
