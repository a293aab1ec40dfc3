"""Infinite and NaN activations through the linear that splits K (33 to 64
rows) and the GEMM: the infinities and NaN of x times the dequantized weight, as
F.linear gives them, in the outliers' columns and beside them."""
import numpy as np
import pytest
import torch

from atlasinfer_amd import _lib
from atlasinfer_amd.integration import atlas_wrappers as AW
from atlasinfer_amd.quant import adaptive_quantizer as AQ
from gpu_ref import make_weights

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
INF, NAN = float("inf"), float("nan")


def _weight(N, K, G, fmt, seed):
    w = torch.from_numpy(make_weights(np.random.default_rng(seed), (N, K), t_dof=3, frac=0.002)).to(DEV)
    q = AQ.quantize_tensor(w, G, 6.0 if G == 64 else 8.0, code_format=fmt)  # few outliers; blocks of 64 hold none past 7.9
    deq = AQ.dequantize_tensor(q, DEV)
    AQ.discard_dequantized(id(q))
    return q, deq


def _x(M, K, deq, q, seed):
    """Rows: finite, an infinity in an outlier's column, in a column without
    outliers, two of them (of either sign), one beside a NaN, all NaN."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    cols = torch.unique(q.outlier_indices % K).tolist()
    plain = next(k for k in range(K) if k not in set(cols))
    x[1, cols[0]] = INF
    x[2, plain] = -INF
    x[3, cols[0]], x[3, cols[-1]] = INF, -INF
    x[4, cols[len(cols) // 2]], x[4, plain] = -INF, INF
    x[5, cols[0]], x[5, K - 1] = INF, NAN
    x[6] = NAN
    x[M - 1, cols] = INF
    return x


def _check(y, x, deq, bias=None):
    # float64 on the host: products and sums in order, nothing padded
    want = x.cpu().double() @ deq.cpu().double().t()
    if bias is not None:
        want = want + bias.cpu().double()
    y = y.cpu().double()
    assert torch.isposinf(want).any() and torch.isneginf(want).any() and torch.isnan(want).any()
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(y), kind(want))
    fin = torch.isfinite(want)
    # one rounding of the output and a worst-case f32 accumulation error
    fx = torch.where(torch.isfinite(x), x, 0).cpu().double()
    bound = 2.0 ** -11 * want.abs() + 2.0 ** -24 + 2.0 ** -20 * (fx.abs() @ deq.cpu().double().abs().t())
    assert ((y - want).abs()[fin] <= bound[fin]).all()


@pytest.mark.parametrize("M", [33, 64])
@pytest.mark.parametrize("N,K,G,fmt", [(48, 4224, -1, "e4m3"), (272, 4096, 128, "int8"), (1040, 4096, 64, "e4m3")])
def test_infinities_stay(N, K, G, fmt, M):
    q, deq = _weight(N, K, G, fmt, N + K)
    x = _x(M, K, deq, q, M)
    bias = torch.randn(N, device=DEV).half()
    codes, tiles = AQ.kernel_codes(q, DEV), AQ.outlier_tiles(q, DEV)
    assert int(tiles[2]) <= 20 and int(_lib.load().aq_qlinear_decode_workspace_size(M, N, K)) > 0  # takes the split-K linear
    y = AW.qlinear(x, q, bias, codes=codes, tiles=tiles)
    _check(y, x, deq, bias)
    assert torch.equal(AW.qlinear_decode(x, [q], [bias], [codes], tiles=[tiles])[0].view(torch.int16),
                       y.view(torch.int16))


@pytest.mark.parametrize("M", [49, 130])
@pytest.mark.parametrize("G,fmt", [(-1, "e4m3"), (128, "int8")])
def test_infinities_stay_in_the_gemm(G, fmt, M):
    q, deq = _weight(272, 1024, G, fmt, 3)
    x = _x(M, 1024, deq, q, M)
    _check(AW.qlinear(x, q, None, codes=AQ.kernel_codes(q, DEV), tiles=AQ.outlier_tiles(q, DEV)), x, deq)


def test_infinities_stay_in_groups():
    """Members of different sizes, whose rows end inside waves of the sum."""
    M, K = 40, 4096
    ws = [_weight(n, K, 128, "e4m3", n) for n in (528, 16, 160)]
    x = _x(M, K, ws[0][1], ws[0][0], 1)
    for y, (_, deq) in zip(AW.qlinear_grouped(x, [w[0] for w in ws]), ws):
        _check(y, x, deq)


def test_weights_that_are_not_finite():
    """A block scale of infinity, with every kind of x."""
    N, K, M = 64, 4096, 33
    q, _ = _weight(N, K, 128, "e4m3", 5)
    q.scale_factors[7] = INF
    deq = AQ.dequantize_tensor(q, DEV)
    AQ.discard_dequantized(id(q))
    x = _x(M, K, deq, q, 2)
    want = x.cpu().double() @ deq.cpu().double().t()
    y = AW.qlinear(x, q, None, codes=AQ.kernel_codes(q, DEV), tiles=AQ.outlier_tiles(q, DEV)).cpu().double()
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(y), kind(want))
