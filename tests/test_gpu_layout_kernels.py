"""The layout kernels through the C ABI against numpy, at the edges of their
spans (8192 elements a workgroup), runs (8 elements a thread) and tiles:
compacted stream <-> dense codes, dequantize from dense, tiled and compacted
codes.  Every result is a byte or the one rounding of an fp16 product, so all
comparisons are exact."""
import numpy as np
import pytest
import torch

from atlasinfer_amd import _lib
from gpu_ref import tile_np

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _call(name, *args):
    _lib.check(getattr(_lib.load(), name)(*args, _lib.stream_of(DEV)), name)


def _e4m3(c):
    """fp16 values of E4M3 codes 0x00..0x7E and their negatives."""
    return torch.from_numpy(c).view(torch.float8_e4m3fn).to(torch.float16).numpy()


def _problem(numel, G, density, fmt, seed):
    rng = np.random.default_rng(seed)
    padded = -(-numel // G) * G
    codes = rng.integers(0, 256, padded, dtype=np.uint8)
    if fmt == _lib.FMT_E4M3:
        codes[(codes & 0x7F) == 0x7F] = 0x80  # no NaN codes; -0 among them
    out = rng.random(padded) < density
    codes[out] = 0
    idx = np.flatnonzero(out).astype(np.int64)
    vals = (rng.standard_normal(idx.size) * 30).astype(np.float16)
    scales = (rng.random(padded // G) * 0.01 + 1e-6).astype(np.float16)
    v = codes.view(np.int8).astype(np.float16) if fmt == _lib.FMT_INT8 else _e4m3(codes)
    want = (v * np.repeat(scales, G))[:numel]
    inside = idx < numel
    want[idx[inside]] = vals[inside]
    return padded, codes, idx, vals, scales, want


# (numel, G): around one run, one span and several; blocks inside, across and
# larger than runs and spans; a padded tail
SIZES = [(1, 1), (7, 3), (8, 8), (9, 5), (1000, 100), (8191, 1), (8192, 128), (8193, 7), (16384, 20000), (24569, 24),
         (40000, 129), (100003, 64)]


@pytest.mark.parametrize("density", [0.0, 0.004, 0.5, 1.0])
@pytest.mark.parametrize("numel,G", SIZES)
def test_stream_round_trip_and_dequantize(numel, G, density):
    padded, codes, idx, vals, scales, want = _problem(numel, G, density, _lib.FMT_INT8, numel + G)
    keep = np.ones(padded, bool)
    keep[idx] = False
    stream = codes[keep]
    didx, dvals, dsc, dcodes = _dev(idx), _dev(vals), _dev(scales), _dev(codes)
    p = _lib.ptr
    # one byte of guard behind the stream: the compaction writes no further
    got = torch.full((stream.size + 1,), 0x5A, dtype=torch.uint8, device=DEV)
    _call("aq_compact_codes", dcodes.data_ptr(), padded, p(didx), idx.size, got.data_ptr())
    assert np.array_equal(got.cpu().numpy(), np.append(stream, np.uint8(0x5A)))
    dense = torch.full((padded + 1,), 0x5A, dtype=torch.uint8, device=DEV)
    _call("aq_expand_codes", got.data_ptr(), padded, p(didx), idx.size, dense.data_ptr())
    assert np.array_equal(dense.cpu().numpy(), np.append(codes, np.uint8(0x5A)))
    for shift in (0, 1):  # an output 16-byte aligned, and one that is not
        y = torch.zeros(numel + 9, dtype=torch.float16, device=DEV)
        _call("aq_dequantize_stream", got.data_ptr(), dsc.data_ptr(), numel, G, p(didx), p(dvals), idx.size,
              y.data_ptr() + 2 * shift)
        y = y.cpu().numpy()
        assert np.array_equal(y[shift:shift + numel].view(np.uint16), want.view(np.uint16))
        assert not y[:shift].any() and not y[shift + numel:].any()


@pytest.mark.parametrize("fmt", [_lib.FMT_INT8, _lib.FMT_E4M3])
@pytest.mark.parametrize("numel,G", SIZES)
def test_dequantize_dense(numel, G, fmt):
    padded, codes, idx, vals, scales, want = _problem(numel, G, 0.01, fmt, numel + 3 * G)
    didx, dvals, dsc = _dev(idx), _dev(vals), _dev(scales)
    for cshift, yshift in ((0, 0), (3, 1)):  # aligned codes and output, and neither
        dcodes = _dev(np.concatenate([np.zeros(cshift, np.uint8), codes]))
        y = torch.zeros(numel + 9, dtype=torch.float16, device=DEV)
        _call("aq_dequantize", dcodes.data_ptr() + cshift, dsc.data_ptr(), numel, G, fmt, numel, _lib.LAYOUT_FLAT,
              _lib.ptr(didx), _lib.ptr(dvals), idx.size, y.data_ptr() + 2 * yshift)
        y = y.cpu().numpy()
        assert np.array_equal(y[yshift:yshift + numel].view(np.uint16), want.view(np.uint16))
        assert not y[yshift + numel:].any()


# rows, cols, G: one tile, a band of 8 tiles less and more one, blocks that
# divide the rows, and blocks that do not (any size the flat elements allow)
@pytest.mark.parametrize("fmt", [_lib.FMT_INT8, _lib.FMT_E4M3])
@pytest.mark.parametrize("rows,cols,G", [(16, 128, 128), (48, 896, 64), (32, 1152, 1152), (16, 2176, 8),
                                         (32, 1024, 40), (64, 384, 20000), (16, 256, 3)])
def test_dequantize_tiled(rows, cols, G, fmt):
    numel = rows * cols
    padded, codes, idx, vals, scales, want = _problem(numel, G, 0.01, fmt, rows + cols + G)
    tiled = _dev(tile_np(codes[:numel], rows, cols))
    inside = idx < numel
    didx, dvals, dsc = _dev(idx[inside]), _dev(vals[inside]), _dev(scales)
    for shift in (0, 1):
        y = torch.zeros(numel + 9, dtype=torch.float16, device=DEV)
        _call("aq_dequantize", tiled.data_ptr(), dsc.data_ptr(), numel, G, fmt, cols, _lib.LAYOUT_TILED,
              _lib.ptr(didx), _lib.ptr(dvals), int(inside.sum()), y.data_ptr() + 2 * shift)
        assert np.array_equal(y.cpu().numpy()[shift:shift + numel].view(np.uint16), want.view(np.uint16))


def _lists(padded):
    """Index lists that do not ascend: repeats, descending, shuffled, past either end."""
    rng = np.random.default_rng(padded)
    n = padded // 2
    return [np.full(n, 5), np.arange(n)[::-1], rng.permutation(padded)[:n], rng.integers(0, padded, n),
            np.full(n, padded + 99), np.full(n, -3), np.sort(rng.integers(-padded, 2 * padded, n))]


@pytest.mark.parametrize("which", range(7))
@pytest.mark.parametrize("padded", [16384, 24576 + 13])
def test_lists_that_do_not_ascend_stay_inside(padded, which):
    """The codes are undefined then, but guards of a list's length on both
    sides of the buffers are neither written nor read."""
    idx = np.ascontiguousarray(_lists(padded)[which]).astype(np.int64)
    nnz, didx = idx.size, _dev(idx)
    left = padded - nnz
    dense, stream, y = (torch.full((3 * padded,), 0x5A, dtype=t, device=DEV)
                        for t in (torch.uint8, torch.uint8, torch.float16))
    dense[padded:2 * padded] = 7
    _call("aq_compact_codes", dense[padded:].data_ptr(), padded, didx.data_ptr(), nnz, stream[padded:].data_ptr())
    assert (stream[:padded] == 0x5A).all() and (stream[padded + left:] == 0x5A).all()
    stream[padded:padded + left] = 7
    _call("aq_expand_codes", stream[padded:].data_ptr(), padded, didx.data_ptr(), nnz, dense[padded:].data_ptr())
    assert (dense[:padded] == 0x5A).all() and (dense[2 * padded:] == 0x5A).all()
    got = dense[padded:2 * padded]
    assert ((got == 0) | (got == 7)).all()
    sc, vals = torch.ones(1, dtype=torch.float16, device=DEV), torch.full((nnz,), 3.0, dtype=torch.float16, device=DEV)
    _call("aq_dequantize_stream", stream[padded:].data_ptr(), sc.data_ptr(), padded, padded, didx.data_ptr(),
          vals.data_ptr(), nnz, y[padded:].data_ptr())
    assert (y[:padded] == 0x5A).all() and (y[2 * padded:] == 0x5A).all()
    got = y[padded:2 * padded]
    assert ((got == 0) | (got == 7) | (got == 3)).all()
