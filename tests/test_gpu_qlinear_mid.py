"""qlinear_decode and plain linears at 33 to 64 rows, where some grids split K
over workgroups (aq_qlinear_decode_workspace_size says which): against the
float64 product of x and the dequantized weight, with every split the workspace
allows (the parts' sums differ in order only), the decode epilogue, ragged last
units, odd part lengths and crowded blocks."""
import ctypes

import numpy as np
import pytest
import torch

from atlasinfer_amd import _lib
from atlasinfer_amd.integration import atlas_wrappers as AW
from atlasinfer_amd.quant import adaptive_quantizer as AQ
from gpu_ref import make_weights

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _weight(N, K, G, fmt, seed, frac=0.002, thr=3.0):
    rng = np.random.default_rng(seed)
    w = torch.from_numpy(make_weights(rng, (N, K), t_dof=3, frac=frac)).to(DEV)
    q = AQ.quantize_tensor(w, G, thr, code_format=fmt)
    deq = AQ.dequantize_tensor(q, DEV).double()
    AQ.discard_dequantized(id(q))
    return q, deq


def _x(M, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(M, K, generator=g, device=DEV).half()


def _close(y, x, deq, bias=None):
    want = x.double() @ deq.t()
    if bias is not None:
        want = want + bias.double()
    ulp = torch.from_numpy(np.spacing(np.abs(want.cpu().numpy()).astype(np.float16)).astype(np.float64)).to(DEV)
    # one rounding of the output and a worst-case f32 accumulation error
    bound = ulp + 2.0 ** -20 * (x.double().abs() @ deq.abs().t())
    assert ((y.double() - want).abs() <= bound).all()


# rows, cols, block, rows of x, format: units of 128 columns that end inside
# the matrix (48, 272), chunks that do not divide by the parts (7, 11, 23),
# scales per row, per chunk and finer, both row-group counts
@pytest.mark.parametrize("N,K,G,M,fmt", [(48, 896, -1, 33, "e4m3"), (272, 1408, 128, 48, "e4m3"),
                                         (4096, 2944, 64, 49, "e4m3"), (1024, 4096, 256, 64, "int8"),
                                         (256, 9472, -1, 64, "e4m3"), (12304, 1024, -1, 40, "e4m3"),
                                         # the decode rule's own side: 33, 35, 21, 96 and 17 chunks
                                         (48, 4224, -1, 33, "e4m3"), (272, 4480, 128, 48, "e4m3"),
                                         (4096, 2688, 64, 49, "e4m3"), (4112, 12288, -1, 40, "int8"),
                                         (24592, 2176, 128, 64, "e4m3"), (32784, 2048, -1, 49, "e4m3")])
def test_mid_matches_dequantized_product(N, K, G, M, fmt):
    q, deq = _weight(N, K, G, fmt, N + K)
    x = _x(M, K, M)
    bias = _x(1, N, 5)[0]
    res = _x(M, N, 6)
    codes, tiles = [AQ.kernel_codes(q, DEV)], [AQ.outlier_tiles(q, DEV)]
    y = AW.qlinear_decode(x, [q], [bias], codes, tiles=tiles)[0]
    _close(y, x, deq, bias)
    z = AW.qlinear_decode(x, [q], [bias], codes, tiles=tiles, relu=[1], residuals=[res])[0]
    assert torch.equal(z, torch.relu(y) + res)
    assert torch.equal(y, AW.qlinear_decode(x, [q], [bias], codes, tiles=tiles)[0])  # deterministic


def test_mid_every_split():
    """A workspace of s parts' bytes, less one, or none: fewer parts, same result to f32 rounding."""
    N, K, M = 512, 3200, 64
    q, deq = _weight(N, K, 128, "e4m3", 3)
    x = _x(M, K, 1)
    L, arr = _lib.load(), _lib.ptr_array
    tp, te, _ = AQ.outlier_tiles(q, DEV)
    full = int(L.aq_qlinear_decode_workspace_size(M, N, K))
    assert full >= 2 * M * N * 4 and full % (M * N * 4) == 0
    for nbytes in [0] + [p * M * N * 4 - 16 * (p % 2) for p in range(1, full // (M * N * 4) + 1)]:
        ws = torch.full((max(nbytes, 16),), 0xFF, dtype=torch.uint8, device=DEV)  # NaN where nothing is written
        y = torch.empty(M, N, dtype=torch.float16, device=DEV)
        _lib.check(L.aq_qlinear_decode_ws(
            x.data_ptr(), M, K, _lib.FMT_E4M3, 1, arr([N], ctypes.c_int64), arr([q.fp8_data.data_ptr()]),
            arr([q.scale_factors.data_ptr()]), arr([q.block_size], ctypes.c_int64), arr([q.outlier_row_ptr.data_ptr()]),
            arr([q.outlier_cols.data_ptr()]), arr([q.fp16_outliers.data_ptr()]), arr([tp.data_ptr()]),
            arr([te.data_ptr()]), arr([None]), arr([y.data_ptr()]), 0, None, None, None, ctypes.c_float(0), None, None,
            ws.data_ptr() if nbytes else None, nbytes, _lib.stream_of(DEV)), "aq_qlinear_decode_ws")
        _close(y, x, deq)


def _decode_ws(x, q, nbytes):
    """aq_qlinear_decode_ws with a workspace of ``nbytes``."""
    (M, K), N = x.shape, q.original_shape[0]
    L, arr = _lib.load(), _lib.ptr_array
    tp, te, _ = AQ.outlier_tiles(q, DEV)
    codes = AQ.kernel_codes(q, DEV)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=DEV)  # NaN where nothing is written
    y = torch.empty(M, N, dtype=torch.float16, device=DEV)
    _lib.check(L.aq_qlinear_decode_ws(
        x.data_ptr(), M, K, _lib.FORMATS[q.code_format], 1, arr([N], ctypes.c_int64), arr([codes.data_ptr()]),
        arr([q.scale_factors.data_ptr()]), arr([q.block_size], ctypes.c_int64), arr([q.outlier_row_ptr.data_ptr()]),
        arr([q.outlier_cols.data_ptr()]), arr([q.fp16_outliers.data_ptr()]), arr([tp.data_ptr()]),
        arr([te.data_ptr()]), arr([None]), arr([y.data_ptr()]), 0, None, None, None, ctypes.c_float(0), None, None,
        ws.data_ptr(), nbytes, _lib.stream_of(DEV)), "aq_qlinear_decode_ws")
    return y


# two parts of 62 to 66 and of 129 chunks: the registers that hold 64 chunks'
# outlier ranges are filled again on the way, once and twice
@pytest.mark.parametrize("M", [33, 64])
@pytest.mark.parametrize("chunks,G,fmt", [(124, -1, "e4m3"), (126, 128, "int8"), (128, 64, "e4m3"), (130, -1, "e4m3"),
                                          (132, 128, "e4m3"), (258, -1, "int8")])
def test_mid_long_parts(chunks, G, fmt, M):
    N, K = 144, 128 * chunks
    q, deq = _weight(N, K, G, fmt, chunks)
    x = _x(M, K, M)
    _close(_decode_ws(x, q, 2 * M * N * 4), x, deq)


@pytest.mark.parametrize("N,K,M", [(80, 4224, 33), (1616, 4096, 64), (12304, 2048, 50), (16400, 2048, 64)])
def test_mid_pair_is_its_members(N, K, M):
    """gate and up as a pair sum as they do alone: bit for bit aq_silu_mul of the two."""
    (g, _), (u, _) = _weight(N, K, 128, "e4m3", 1), _weight(N, K, 128, "e4m3", 2)
    x = _x(M, K, 2)
    codes = [q.fp8_data.view(torch.uint8) for q in (g, u)]
    assert int(_lib.load().aq_qlinear_decode_workspace_size(M, 2 * N, K)) > 0
    a = AW.qlinear_decode(x, [g, u], [None, None], codes, swiglu_pair=True)[0]
    yg, yu = AW.qlinear_decode(x, [g, u], [None, None], codes)
    want = torch.empty_like(yg)
    _lib.check(_lib.load().aq_silu_mul(yg.data_ptr(), yu.data_ptr(), want.data_ptr(), M * N, _lib.stream_of(DEV)),
               "aq_silu_mul")
    assert torch.equal(a, want)


def test_mid_grouped_and_swiglu_pair():
    """Members of different sizes in one launch; gate and up as a pair, split and not."""
    K, M = 1664, 50
    ws = [_weight(n, K, -1, "e4m3", n) for n in (1040, 256, 16)]
    x = _x(M, K, 2)
    ys = AW.qlinear_decode(x, [w[0] for w in ws], [None] * 3, [w[0].fp8_data.view(torch.uint8) for w in ws])
    for y, (_, deq) in zip(ys, ws):
        _close(y, x, deq)
    for N in (80, 1616, 8208):
        (g, dg), (u, du) = _weight(N, K, 128, "e4m3", 1), _weight(N, K, 128, "e4m3", 2)
        codes = [q.fp8_data.view(torch.uint8) for q in (g, u)]
        a = AW.qlinear_decode(x, [g, u], [None, None], codes, swiglu_pair=True)[0]
        yg, yu = AW.qlinear_decode(x, [g, u], [None, None], codes)
        want = torch.nn.functional.silu(yg.float()).half() * yu
        # silu rounded to fp16 one way or the other, then the product
        ulp = np.spacing(np.abs(want.cpu().numpy()).astype(np.float16)).astype(np.float32)
        assert (np.abs(a.float().cpu().numpy() - want.float().cpu().numpy()) <= 2 * ulp).all()


def test_mid_crowded_blocks():
    """Chunks with more outliers than travel with the codes (8), and more than 64."""
    q, deq = _weight(64, 1024, 128, "e4m3", 9, frac=0.05, thr=1.2)
    assert int(q.outlier_tile_max) > 64
    x = _x(64, 1024, 4)
    y = AW.qlinear_decode(x, [q], [None], [q.fp8_data.view(torch.uint8)])[0]
    _close(y, x, deq)


# plain linears on both sides of the rule (more than 48 rows with K below 4096
# and weights with more than 20 outliers in a block take the GEMM), ragged last
# units, all scale modes
@pytest.mark.parametrize("thr", [3.0, 8.0])
@pytest.mark.parametrize("M", [33, 48, 49, 64])
@pytest.mark.parametrize("N,K,G,fmt", [(48, 1024, -1, "e4m3"), (272, 3968, 128, "int8"), (2064, 4096, 64, "e4m3")])
def test_mid_plain(N, K, G, fmt, M, thr):
    q, deq = _weight(N, K, G, fmt, N + K, thr=thr)
    x, bias = _x(M, K, M), _x(1, N, 5)[0]
    tiles = AQ.outlier_tiles(q, DEV)
    y = AW.qlinear(x, q, bias, codes=AQ.kernel_codes(q, DEV), tiles=tiles)
    _close(y, x, deq, bias)
    if int(tiles[2]) <= 20 and K >= 4096:  # the decode call's sums
        assert torch.equal(y, AW.qlinear_decode(x, [q], [bias], [AQ.kernel_codes(q, DEV)], tiles=[tiles])[0])


@pytest.mark.parametrize("M", [33, 48, 64])
def test_mid_plain_grouped(M):
    """Members of different sizes in one launch."""
    K = 1664
    ws = [_weight(n, K, -1, "e4m3", n, thr=8.0) for n in (1040, 256, 16)]
    x = _x(M, K, 2)
    for y, (_, deq) in zip(AW.qlinear_grouped(x, [w[0] for w in ws]), ws):
        _close(y, x, deq)


@pytest.mark.parametrize("parts", [0, 1, 2, 3])
def test_mid_plain_workspaces(parts):
    """Workspaces too small for two parts leave the call to the GEMM or the GEMV, others limit the split."""
    N, K = 512, 3200
    q, deq = _weight(N, K, 128, "e4m3", 3, thr=8.0)
    tp, te, tmax = AQ.outlier_tiles(q, DEV)
    for M in (40, 64):
        x = _x(M, K, 1)
        nbytes = parts * M * N * 4
        ws = torch.full((max(nbytes, 16),), 0xFF, dtype=torch.uint8, device=DEV)  # NaN where nothing is written
        y = torch.empty(M, N, dtype=torch.float16, device=DEV)
        _lib.check(_lib.load().aq_qlinear(
            x.data_ptr(), M, K, N, q.fp8_data.data_ptr(), q.scale_factors.data_ptr(), q.block_size, _lib.FMT_E4M3,
            q.outlier_row_ptr.data_ptr(), q.outlier_cols.data_ptr(), q.fp16_outliers.data_ptr(), tp.data_ptr(),
            te.data_ptr(), tmax, None, y.data_ptr(), ws.data_ptr() if nbytes else None, nbytes, _lib.stream_of(DEV)),
            "aq_qlinear")
        _close(y, x, deq)
