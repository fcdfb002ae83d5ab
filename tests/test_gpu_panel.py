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

# NUQ_PANEL_SHAPES (nuclis_amd/csrc/panel.h): TG, RG, WR, WK, DEPTH
SHAPES = [(1, 1, 4, 1, 4), (1, 1, 2, 4, 2), (2, 1, 2, 2, 2), (3, 1, 4, 2, 2), (4, 1, 4, 2, 2),
          (4, 1, 2, 2, 2), (4, 1, 4, 1, 2), (4, 2, 4, 1, 2), (6, 2, 4, 1, 2), (8, 2, 4, 1, 2)]


class Plan(ctypes.Structure):
    _fields_ = [("shape", ctypes.c_int), ("full", ctypes.c_uint32), ("tail", ctypes.c_uint32),
                ("splits", ctypes.c_uint32), ("work_floats", ctypes.c_uint64), ("cost", ctypes.c_float)]


class Args(ctypes.Structure):
    _fields_ = [("w", ctypes.c_void_p), ("stride", ctypes.c_uint64), ("rows", ctypes.c_uint32),
                ("columns", ctypes.c_uint32), ("x", ctypes.c_void_p), ("in_stride", ctypes.c_uint64),
                ("y", ctypes.c_void_p), ("out_stride", ctypes.c_uint64), ("tokens", ctypes.c_uint32)]


@pytest.fixture(scope="module")
def backend():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    b = nq.Backend(0)
    yield b
    b.close()


def launch(encoding, args, plan, work):
    import torch
    f = nq.lib()._ZN3nuq12launch_panelEP12ihipStream_tjRKNS_9PanelArgsERKNS_9PanelPlanEPf
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.POINTER(Args), ctypes.POINTER(Plan), ctypes.c_void_p]
    return f(torch.cuda.current_stream().cuda_stream, encoding, ctypes.byref(args), ctypes.byref(plan), work)


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
        args = Args(wg.data_ptr(), w.shape[1], rows, columns, xg.data_ptr(), in_stride, y.data_ptr(), out_stride, tokens)
        assert launch(encoding, args, Plan(shape, full, tail, splits, 0, 0.0), work.data_ptr()) == 0
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert np.isnan(got[:, rows:]).all() and np.isfinite(got[:, :rows]).all()
        check_close(got[check, :rows], want, m, F16_K, f"panel {encoding} shape {shape} splits {splits} tail {tail}")


@pytest.mark.parametrize("splits", [2, 4, 5, 6, 9, 11])
def test_partial_sums_of_any_split_count(backend, splits):
    """The reduction reads four splits at a time: counts around its turns."""
    import torch
    rows, tokens, columns = 136, 33, 256 * 11
    w = nq.quantize(14, gaussian(41, (rows, columns), 0.02))
    x = gaussian(42, (tokens, columns)).astype(np.float16)
    wg, xg = to_gpu(w), to_gpu(x)
    work, y = torch.empty(4 * splits * 32 * 128, device="cuda"), torch.full((tokens, rows), np.nan, device="cuda")
    args = Args(wg.data_ptr(), w.shape[1], rows, columns, xg.data_ptr(), columns, y.data_ptr(), rows, tokens)
    assert launch(14, args, Plan(0, 0, 4, splits, 0, 0.0), work.data_ptr()) == 0
    torch.cuda.synchronize()
    xr = x.astype(np.float32)
    check_close(y.cpu().numpy(), orc.matmul(14, rows, columns, w, xr), mass(14, w, rows, columns, xr), F16_K,
                f"panel {splits} splits")


@pytest.mark.parametrize("encoding,rows,columns,tokens", [(12, 1032, 512, 77), (14, 520, 2304, 300), (8, 4104, 2048, 260),
                                                          (8, 264, 320, 40), (23, 8192, 4096, 8)])
def test_f32_activations_equal_their_f16_rounding(backend, encoding, rows, columns, tokens):
    """The tiles round F32 activations to f16: the same bits as f16 input."""
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
