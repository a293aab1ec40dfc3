"""aq_decode_attention at the edges of its steps (16 positions of D = 128, 32
of 64), chunks, waves and spans, every query-group size, with the cache past
the position full of NaN (it must not be read into a result), against float64."""
import ctypes

import pytest
import torch

from atlasinfer_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _run(B, Hkv, G, D, L, pos, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half()  # noqa: E731
    H = Hkv * G
    q, k, v = rnd(B, H, D), rnd(B, Hkv, D), rnd(B, Hkv, D)
    kc = torch.full((B, Hkv, L, D), float("nan"), dtype=torch.float16, device=DEV)
    vc = torch.full_like(kc, float("nan"))
    kc[:, :, :pos], vc[:, :, :pos] = rnd(B, Hkv, pos, D), rnd(B, Hkv, pos, D)
    before_k, before_v = kc.clone(), vc.clone()
    Lb = _lib.load()
    nb = Lb.aq_decode_attention_workspace(B, H, Hkv, D, L)
    ws = torch.full((max(nb, 16),), 0xFF, dtype=torch.uint8, device=DEV)
    out = torch.empty(B, H, D, dtype=torch.float16, device=DEV)
    p = torch.full((1,), pos, dtype=torch.long, device=DEV)
    scale = D ** -0.5
    _lib.check(Lb.aq_decode_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                                      p.data_ptr(), B, H, Hkv, D, L, ctypes.c_float(scale), ctypes.c_float(1.0), None,
                                      None, ws.data_ptr(), nb, out.data_ptr(), _lib.stream_of(DEV)), "attention")
    before_k[:, :, pos], before_v[:, :, pos] = k, v
    assert torch.equal(kc.view(torch.int16), before_k.view(torch.int16))  # written at pos, nowhere else
    assert torch.equal(vc.view(torch.int16), before_v.view(torch.int16))
    kk = before_k[:, :, :pos + 1].double().repeat_interleave(G, 1)
    vv = before_v[:, :, :pos + 1].double().repeat_interleave(G, 1)
    s = (kk * q.double().unsqueeze(2)).sum(-1)
    w = torch.softmax(s * scale, -1)
    want = (vv * w.unsqueeze(-1)).sum(2)
    # the scores are rounded to fp16 (relative 2^-11, so a weight is off by
    # |s| scale 2^-11 relative), the output once, the sums in f32
    off = (s.abs().amax(-1) * scale * 2.0 ** -11 * 2 + 2.0 ** -10).unsqueeze(-1)
    bound = off * (vv.abs() * w.unsqueeze(-1)).sum(2) + 2.0 ** -11 * want.abs() + 1e-6
    assert ((out.double() - want).abs() <= bound).all(), (out.double() - want).abs().max()


@pytest.mark.parametrize("D,G", [(64, 1), (64, 2), (64, 8), (128, 1), (128, 4), (128, 8)])
@pytest.mark.parametrize("pos", [0, 1, 15, 16, 31, 33, 63, 64, 65, 127, 200, 255])
def test_one_and_few_spans(D, G, pos):
    _run(2, 3, G, D, 256, pos, 100 * D + G + pos)


@pytest.mark.parametrize("B,Hkv,G,D,L,pos", [
    (1, 8, 4, 128, 832, 700),      # one-chunk spans of four waves
    (8, 8, 4, 128, 4160, 4000),    # spans of several chunks, the last one partial
    (8, 8, 4, 128, 4160, 512),     # the last span holds the position alone
    (8, 8, 4, 128, 4160, 4159),
    (3, 2, 1, 64, 5000, 4097),     # 64 spans, waves with one and no step
    (300, 2, 2, 128, 640, 511),    # one span by the number of heads
    (64, 32, 1, 64, 700, 650),
])
def test_long_caches(B, Hkv, G, D, L, pos):
    _run(B, Hkv, G, D, L, pos, pos)


# both sides of the splitting rule's lines, with positions that leave waves
# without a step, or with the position alone
@pytest.mark.parametrize("B,Hkv,G,D,L,poss", [
    (64, 16, 1, 64, 320, (0, 31, 32, 130, 319)),     # 1024 heads: one wave
    (64, 16, 2, 64, 832, (5, 700)),
    (32, 16, 2, 64, 320, (33, 319)),                 # 512 heads, 5 chunks: one wave
    (32, 16, 1, 64, 321, (40, 320)),                 # 6 chunks: four
    (16, 8, 4, 128, 448, (0, 15, 16, 47, 48, 300)),  # 128 heads: one span of four waves
    (127, 1, 4, 128, 448, (16, 300)),                # 127: split
    (1, 4, 8, 64, 192, (31, 32, 190)),               # 8 chunk-units a wave: one span
    (1, 16, 1, 128, 832, (700,)),                    # 13 steps a wave: split
    (25, 8, 1, 64, 4160, (64, 4100)),                # 200 heads: a span longer than the cache
    (8, 8, 4, 128, 1664, (511, 512, 1500)),          # spans of 8 chunks
])
def test_splitting(B, Hkv, G, D, L, poss):
    for pos in poss:
        _run(B, Hkv, G, D, L, pos, pos)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("pos,low", [(40, 32), (700, 650), (4000, 64)])
def test_scores_of_minus_infinity(D, pos, low):
    """The first ``low`` positions' scores overflow fp16 to -inf, for whole
    steps, waves and spans: they weigh nothing, and the rest come out as if
    alone."""
    Hkv, L = 2, 4160
    g = torch.Generator(device=DEV).manual_seed(pos + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half()  # noqa: E731
    q = rnd(1, Hkv, D).abs() + 1.0
    kc, vc, k, v = rnd(1, Hkv, L, D) * 0.1, rnd(1, Hkv, L, D), rnd(1, Hkv, D) * 0.1, rnd(1, Hkv, D)
    kc[:, :, :low] = -60000.0  # products below -60000 D
    Lb = _lib.load()
    nb = Lb.aq_decode_attention_workspace(1, Hkv, Hkv, D, L)
    ws = torch.full((max(nb, 16),), 0xFF, dtype=torch.uint8, device=DEV)
    out = torch.empty(1, Hkv, D, dtype=torch.float16, device=DEV)
    p = torch.full((1,), pos, dtype=torch.long, device=DEV)
    scale = D ** -0.5
    _lib.check(Lb.aq_decode_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                                      p.data_ptr(), 1, Hkv, Hkv, D, L, ctypes.c_float(scale), ctypes.c_float(1.0), None,
                                      None, ws.data_ptr(), nb, out.data_ptr(), _lib.stream_of(DEV)), "attention")
    s = (kc[:, :, low:pos + 1].double() * q.double().unsqueeze(2)).sum(-1)
    vv = vc[:, :, low:pos + 1].double()
    w = torch.softmax(s * scale, -1)
    want = (vv * w.unsqueeze(-1)).sum(2)
    # as in _run
    off = (s.abs().amax(-1) * scale * 2.0 ** -11 * 2 + 2.0 ** -10).unsqueeze(-1)
    bound = off * (vv.abs() * w.unsqueeze(-1)).sum(2) + 2.0 ** -11 * want.abs() + 1e-6
    assert ((out.double() - want).abs() <= bound).all()
