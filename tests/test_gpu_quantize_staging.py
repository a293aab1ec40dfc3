"""The quantize kernel's outlier staging, shared by the blocks of a wave: the
flat lists (aq_quantize_finish) and the block lists (aq_quantize_finish_tiles)
read back from it equal lists built with numpy from the oracle's outliers, for
every team shape, for staging units that cross rows and tile rows or end past
the last block, and for tile rows with few, many and very many entries."""
import numpy as np
import pytest
import torch

from atlasinfer_amd import _lib
from gpu_ref import make_weights

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _tiles(idx, vals, N, K):
    """(tile_ptr, tile_ent) of ascending flat outliers, block by block."""
    r, c = idx // K, idx % K
    nch = K // 64
    block = (r // 16) * nch + c // 64
    order = np.lexsort((c, r, block))
    ptr = np.zeros((N // 16) * nch + 1, np.int64)
    np.add.at(ptr, block + 1, 1)
    ent = (vals.view(np.uint16).astype(np.uint32) << 16) | ((r % 16) << 6 | c % 64).astype(np.uint32)
    return np.cumsum(ptr).astype(np.int32), ent[order]


# rows, cols, G, threshold: teams of 1 to 1024 threads; units of several
# blocks that end inside the weight's last tile row, cross rows (192 / 64,
# 320 / 64: 48 and 80 blocks a tile row in units of 32) or hold one row each
CASES = [(32, 64, 8, 1.5), (48, 64, 16, 1.5), (16, 96 * 2, 32, 2.0), (48, 192, 64, 2.0), (80, 320, 64, 2.0),
         (16, 64, 64, 2.0), (48, 128, 128, 2.0), (32, 1152, 128, 2.0), (16, 768, 256, 2.0), (16, 512, 512, 2.0),
         (48, 1024, 1024, 2.0), (16, 1984, 1984, 2.5), (32, 2304, 2304, 2.5), (16, 8192, 8192, 2.5),
         (16, 14336, 14336, 2.5), (16, 20032, 20032, 2.5),
         # entries a tile row: about 500, 1000, and past the registers (12 000)
         (64, 4096, 128, 2.6), (32, 4096, 128, 2.3), (32, 4096, 4096, 2.5), (16, 4096, 128, 1.2)]


@pytest.mark.parametrize("N,K,G,thr", CASES)
def test_lists_from_the_stage(oracle, N, K, G, thr):
    rng = np.random.default_rng(N * K + G)
    w = make_weights(rng, (N, K), t_dof=3, frac=0.01)
    ref = oracle.quantize(w, G, thr, oracle.FMT_E4M3)
    idx, vals = ref["outlier_indices"], ref["fp16_outliers"]
    L, s, ck = _lib.load(), _lib.stream_of(DEV), _lib.check
    x = torch.from_numpy(w).to(DEV)
    numel, nb = N * K, N * K // G
    u8 = lambda n: torch.empty(n, dtype=torch.uint8, device=DEV)  # noqa: E731
    i32 = lambda n: torch.full((n,), -1, dtype=torch.int32, device=DEV)  # noqa: E731
    codes, scales, off = u8(numel), torch.empty(nb, dtype=torch.float16, device=DEV), i32(nb + 1)
    ws = u8(int(L.aq_quantize_workspace_size(numel, G)))
    ck(L.aq_quantize(x.data_ptr(), numel, G, int(np.float16(thr).view(np.uint16)), _lib.FMT_E4M3, K, _lib.LAYOUT_FLAT,
                     codes.data_ptr(), scales.data_ptr(), off.data_ptr(), ws.data_ptr(), ws.numel(), s), "aq_quantize")
    nnz = int(off[-1].item())
    assert nnz == idx.size
    tptr, tent, tmax = i32((N // 16) * (K // 64) + 1), i32(nnz + 64), torch.zeros(1, dtype=torch.int32, device=DEV)
    want_ptr, want_ent = _tiles(idx, vals, N, K)
    for tiles in (False, True):
        fi = torch.full((nnz,), -1, dtype=torch.int64, device=DEV)
        va, co = torch.empty(nnz, dtype=torch.float16, device=DEV), i32(nnz)
        args = (numel, G, K, off.data_ptr(), nnz, ws.data_ptr(), ws.numel(), _lib.ptr(fi), _lib.ptr(va), _lib.ptr(co))
        if tiles:
            ck(L.aq_quantize_finish_tiles(*args, tptr.data_ptr(), tent.data_ptr(), tmax.data_ptr(), s), "finish_tiles")
        else:
            ck(L.aq_quantize_finish(*args, s), "finish")
        assert np.array_equal(fi.cpu().numpy(), idx)
        assert np.array_equal(va.cpu().numpy().view(np.uint16), vals.view(np.uint16))
        assert np.array_equal(co.cpu().numpy(), (idx % K).astype(np.int32))
    assert np.array_equal(tptr.cpu().numpy(), want_ptr)
    assert np.array_equal(tent.cpu().numpy().view(np.uint32)[:nnz], want_ent)
    assert not tent.cpu().numpy()[nnz:].any()
    assert int(tmax.item()) == int(np.diff(want_ptr).max(initial=0))
