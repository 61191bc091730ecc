"""Prefill attention kernel forms against float64: every form of
the launcher at its edges -- partial last blocks and key tiles, KV heads with 1 to
16 query heads, every head size, INT8 and FP16 caches, windows, padded cache
heads -- V scales beyond the fp16-safe bound of the lazily moved softmax
reference, and references that move in a state's later tiles.  Bar: the output is fp16 (one rounding, 2^-11 of the value) of fp32
sums of ~22-bit probability products; 1e-3 of the largest output plus one fp16
ulp of the value, the bar of the other attention tests."""
import numpy as np
import pytest
import torch

import jllm
import synth
from gpu_util import f16_to_f64, from_dev, print_case, to_dev

pytestmark = pytest.mark.gpu


def _want(q, k, v, start, window, scale):
    """q [N, H, hd], k / v [ctx, KV, hd] in float64."""
    N, H, hd = q.shape
    ctx, KV = k.shape[0], k.shape[1]
    pos, key = np.arange(start, start + N)[:, None], np.arange(ctx)[None, :]
    dead = key > pos
    if window:
        dead |= key <= pos - window
    out = np.empty_like(q)
    for h in range(H):
        g = h // (H // KV)
        s = np.where(dead, -np.inf, q[:, h] @ k[:, g].T * scale)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = (p / p.sum(1, keepdims=True)) @ v[:, g]
    return out


@pytest.mark.parametrize("H,KV,hd,pad,int8,N,start,window,vs_mul", [
    (32, 8, 128, 0, True, 1, 0, 0, 1.0),            # one key
    (32, 8, 128, 0, True, 7, 25, 0, 1.0),           # one partial block, keys end inside a tile
    (32, 8, 128, 0, True, 256, 33, 0, 1.0),         # 256 blocks: 32 columns
    (32, 8, 128, 0, True, 257, 0, 0, 1.0),          # 257 blocks: 64 columns
    (32, 8, 128, 0, True, 300, 724, 0, 1.0),        # 64 columns, 1024 keys
    (32, 8, 128, 0, True, 300, 725, 0, 1.0),        # a partial last tile
    (32, 8, 128, 0, False, 261, 800, 0, 1.0),       # the same form, fp16 cache
    (32, 8, 128, 0, True, 263, 900, 100, 1.0),      # window: short key ranges
    (32, 8, 128, 0, True, 261, 1200, 1100, 1.0),    # window: long key ranges
    (32, 8, 128, 0, True, 40, 100, 0, 3e4),         # V scales beyond AP_VS_MAX (values near the fp16 limit), one tile per wave
    (8, 8, 64, 0, True, 70, 11, 0, 1.0),
    (12, 4, 96, 0, True, 50, 60, 0, 1.0),           # 3 heads per KV head: 30 of 32 columns live
    (12, 4, 96, 0, False, 50, 60, 20, 1.0),
    (32, 2, 32, 0, True, 9, 40, 0, 1.0),            # 16 heads per KV head: 2 tokens a block
    (8, 2, 32, 0, False, 33, 31, 0, 1.0),
    (16, 2, 128, 32, True, 20, 50, 0, 1.0),         # cache heads wider than the head
    (8, 2, 64, 0, False, 64, 64, 0, 1.0),
])
def test_prefill_attention_forms(dev, H, KV, hd, pad, int8, N, start, window, vs_mul):
    print_case("attn_prefill_form", H, KV, hd, pad, int8, N, start, window, vs_mul)
    g = synth.rng(H * 1000 + hd + N + start)
    ctx, chd, scale = start + N, hd + pad, 1.0 / np.sqrt(hd)
    q = synth.x_f16(g, (N, H, hd))
    out = torch.empty(N * H * hd, dtype=torch.int16, device=dev)
    if int8:
        k, v = synth.kv_int8(g, ctx, KV, chd), synth.kv_int8(g, ctx, KV, chd)
        ks, vs = synth.kv_scales(g, ctx, KV), synth.kv_scales(g, ctx, KV) * np.float32(vs_mul)
        vs = np.minimum(vs, np.float32(500.0)) if vs_mul == 1.0 else np.minimum(vs, np.float32(4000.0))
        if vs_mul != 1.0:
            v = np.clip(v, -12, 12)                  # |v * vs| <= 48000 stays an fp16 number
        args = [to_dev(k), to_dev(v), to_dev(ks), to_dev(vs)]
        kf, vf = k[..., :hd] * ks[..., None].astype(np.float64), v[..., :hd] * vs[..., None].astype(np.float64)
    else:
        kh = (g.standard_normal((ctx, KV, chd)) * 0.5).astype(np.float16)
        vh = g.standard_normal((ctx, KV, chd)).astype(np.float16)
        args = [to_dev(kh.view(np.uint16)), to_dev(vh.view(np.uint16)), None, None]
        kf, vf = kh[..., :hd].astype(np.float64), vh[..., :hd].astype(np.float64)
    jllm.call("jllm_hip_flash_attention_prefill_batched", out, to_dev(q), args[0], args[1], H, KV, hd, chd, N, start,
              scale, int(int8), args[2], args[3], window)
    got = f16_to_f64(from_dev(out, np.uint16)).reshape(N, H, hd)
    want = _want(f16_to_f64(q).reshape(N, H, hd), kf, vf, start, window, scale)
    err = np.abs(got - want)
    assert np.all(err <= 1e-3 * np.abs(want).max() + np.abs(want) * 2 ** -10), float(err.max())


@pytest.mark.parametrize("hd", [32, 64, 96, 128])
@pytest.mark.parametrize("N,start", [(20, 700), (300, 200), (300, 900)])    # 32 columns, 64 columns
@pytest.mark.parametrize("with_ks,with_vs", [(False, False), (True, False), (False, True)])
def test_prefill_attention_without_scales(dev, hd, N, start, with_ks, with_vs):
    """INT8 caches whose k_scales and / or v_scales are NULL (= 1.0), several key
    tiles per wave: the kernel's waits count its loads, so a call without scale
    pointers has to issue as many as one with them."""
    print_case("attn_prefill_no_scales", hd, N, start, with_ks, with_vs)
    H, KV = 32, 8
    g = synth.rng(hd + N + start)
    ctx = start + N
    q = synth.x_f16(g, (N, H, hd))
    # without scales K codes of -1, 0, 1: scores of order 1, so that every key counts
    k = synth.kv_int8(g, ctx, KV, hd) if with_ks else g.integers(-1, 2, size=(ctx, KV, hd), dtype=np.int8)
    v = synth.kv_int8(g, ctx, KV, hd)
    ks, vs = synth.kv_scales(g, ctx, KV), synth.kv_scales(g, ctx, KV)
    scale = 1.0 / np.sqrt(hd)
    out = torch.empty(N * H * hd, dtype=torch.int16, device=dev)
    jllm.call("jllm_hip_flash_attention_prefill_batched", out, to_dev(q), to_dev(k), to_dev(v), H, KV, hd, hd, N, start,
              scale, 1, to_dev(ks) if with_ks else None, to_dev(vs) if with_vs else None, 0)
    got = f16_to_f64(from_dev(out, np.uint16)).reshape(N, H, hd)
    kf = k.astype(np.float64) * (ks[..., None].astype(np.float64) if with_ks else 1.0)
    vf = v.astype(np.float64) * (vs[..., None].astype(np.float64) if with_vs else 1.0)
    want = _want(f16_to_f64(q).reshape(N, H, hd), kf, vf, start, 0, scale)
    err = np.abs(got - want)
    assert np.all(err <= 1e-3 * np.abs(want).max() + np.abs(want) * 2 ** -10), float(err.max())


@pytest.mark.parametrize("H,KV,hd,int8,big_vs", [
    (32, 8, 128, True, False),
    (32, 8, 128, True, True),           # single V scales beyond AP_VS_MAX
    (32, 8, 128, False, False),
    (12, 4, 96, True, False),           # blocks of 10 and 21 tokens
    (8, 2, 64, True, False),
    (32, 32, 32, False, False),
])
def test_prefill_attention_bits_do_not_depend_on_the_cut(dev, H, KV, hd, int8, big_vs):
    """A prompt of 1300 tokens in one call and cut into calls that take every form
    of the launcher at every key range: the same bits, whichever form a token's
    call takes."""
    print_case("attn_prefill_cut", H, KV, hd, int8, big_vs)
    g = synth.rng(H + hd)
    T = 1300
    q = to_dev(synth.x_f16(g, (T, H, hd)))
    ks = vs = None
    if int8:
        k, v = synth.kv_int8(g, T, KV, hd), synth.kv_int8(g, T, KV, hd)
        ks, vs = synth.kv_scales(g, T, KV), synth.kv_scales(g, T, KV)
        if big_vs:
            vs[::37] = 2000.0
            v = np.clip(v, -12, 12)
        ks, vs = to_dev(ks), to_dev(vs)
    else:
        k, v = (g.standard_normal((T, KV, hd)).astype(np.float16).view(np.uint16) for _ in range(2))
    k, v = to_dev(k), to_dev(v)
    q = q.view(T, H * hd)
    want = None
    for cut in ([1300], [512, 512, 276], [256] * 5 + [20], [100] * 13, [505, 795], [509, 30, 761], [511, 1, 700, 88]):
        out = torch.zeros_like(q)
        pos = 0
        for n in cut:
            jllm.call("jllm_hip_flash_attention_prefill_batched", out[pos:pos + n], q[pos:pos + n], k, v, H, KV, hd, hd,
                      n, pos, 1.0 / np.sqrt(hd), int(int8), ks, vs, 0)
            pos += n
        assert pos == T
        got = from_dev(out, np.uint16)
        if want is None:
            want = got
        assert np.array_equal(got, want), cut


SLACK, STATES, TILE = 6.0, 8, 32      # AP_SLACK, AP_WAVES (a state each) and the keys of a tile


def _replay(s2, vs, slack=SLACK):
    """The lazily moved reference of one column over its base-2 scores: how often a
    state's reference moved after its first tile, and the largest p * vs."""
    moves, top = 0, 0.0
    for u in range(STATES):
        ref = None
        for p0 in range(u * TILE, len(s2), STATES * TILE):
            t = s2[p0:p0 + TILE]
            if ref is None:
                ref = t.max()
            elif t.max() > ref + slack:
                ref, moves = t.max(), moves + 1
            top = max(top, float((np.exp2(t - ref) * vs[p0:p0 + TILE]).max()))
    return moves, top


# (N, start) on 32 / 8 heads: 32 columns, 64 columns
FORMS = [(20, 1100), (300, 724), (300, 1100)]


@pytest.mark.parametrize("N,start", FORMS)
def test_prefill_attention_v_scales_under_a_lagging_reference(dev, N, start):
    """V scales above AP_VS_MAX where a state's later tiles exceed its reference by
    less than AP_SLACK: with the reference left behind, p * vs would pass the fp16
    range (checked on the inputs), so these tiles have to take the exact maximum."""
    print_case("attn_prefill_vs_lag", N, start)
    H, KV, hd = 32, 8, 128
    g = synth.rng(N + start)
    ctx, scale = start + N, 1.0 / np.sqrt(hd)
    q = (0.5 * (1.0 + 0.05 * g.standard_normal((N, H, hd)))).astype(np.float16)
    k = (64 + g.integers(-8, 9, size=(ctx, KV, hd))).astype(np.int8)
    # base-2 scores by the tile's place in its state: 0, then 5.5 (behind by less
    # than the slack), 5, 11 (moves), 5, ...
    target = np.array([0.02, 5.5, 5.0, 11.0, 5.0, 11.2])[np.arange(ctx) // (TILE * STATES)]
    ks = np.repeat((target * np.log(2.0) / (0.5 * 64 * hd * scale)).astype(np.float32)[:, None], KV, 1)
    v = g.integers(-12, 13, size=(ctx, KV, hd), dtype=np.int8)
    vs = (2000.0 + 2000.0 * g.random((ctx, KV))).astype(np.float32)           # |v * vs| <= 48000
    kf = k * ks[..., None].astype(np.float64)
    s2 = kf[:, 0] @ q[-1, 0].astype(np.float64) * scale / np.log(2.0)
    assert _replay(s2, vs[:, 0])[1] > 65504.0 and _replay(s2, vs[:, 0], 0.0)[1] < 65504.0
    out = torch.empty(N * H * hd, dtype=torch.int16, device=dev)
    jllm.call("jllm_hip_flash_attention_prefill_batched", out, to_dev(q.view(np.uint16)), to_dev(k), to_dev(v), H, KV, hd,
              hd, N, start, scale, 1, to_dev(ks), to_dev(vs), 0)
    got = f16_to_f64(from_dev(out, np.uint16)).reshape(N, H, hd)
    want = _want(q.astype(np.float64), kf, v * vs[..., None].astype(np.float64), start, 0, scale)
    err = np.abs(got - want)
    assert np.all(err <= 1e-3 * np.abs(want).max() + np.abs(want) * 2 ** -10), float(err.max())


@pytest.mark.parametrize("N,start", FORMS)
@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("hd", [32, 64, 96, 128])
def test_prefill_attention_moved_reference(dev, hd, int8, N, start):
    """Several tiles per state, whose maxima grow by more than 2^AP_SLACK from one to
    the next (checked on the inputs) and fall again: the accumulators are rescaled
    in mid-run and the K / V buffers reused, at every head size and cache type."""
    print_case("attn_prefill_moved", hd, int8, N, start)
    H, KV = 32, 8
    g = synth.rng(hd + N + start)
    ctx, scale = start + N, 1.0 / np.sqrt(hd)
    q = g.standard_normal((N, H, hd)).astype(np.float16)
    grow = np.array([1.0, 5.0, 2.0, 9.0, 3.0, 16.0])[np.arange(ctx) // (TILE * STATES)][:, None, None]
    kr, vr = g.standard_normal((ctx, KV, hd)) * grow, g.standard_normal((ctx, KV, hd))
    if int8:
        ks, vs = (np.abs(a).max(-1).astype(np.float32) / np.float32(127) for a in (kr, vr))
        k, v = (np.rint(a / b[..., None]).astype(np.int8) for a, b in ((kr, ks), (vr, vs)))
        kf, vf = k * ks[..., None].astype(np.float64), v * vs[..., None].astype(np.float64)
        args = [to_dev(k), to_dev(v), to_dev(ks), to_dev(vs)]
    else:
        k, v = kr.astype(np.float16), vr.astype(np.float16)
        kf, vf = k.astype(np.float64), v.astype(np.float64)
        args = [to_dev(k.view(np.uint16)), to_dev(v.view(np.uint16)), None, None]
    s2 = kf[:, 0] @ q[-1, 0].astype(np.float64) * scale / np.log(2.0)
    assert _replay(s2, np.ones(ctx))[0] >= STATES
    out = torch.empty(N * H * hd, dtype=torch.int16, device=dev)
    jllm.call("jllm_hip_flash_attention_prefill_batched", out, to_dev(q.view(np.uint16)), args[0], args[1], H, KV, hd, hd,
              N, start, scale, int(int8), args[2], args[3], 0)
    got = f16_to_f64(from_dev(out, np.uint16)).reshape(N, H, hd)
    want = _want(q.astype(np.float64), kf, vf, start, 0, scale)
    err = np.abs(got - want)
    assert np.all(err <= 1e-3 * np.abs(want).max() + np.abs(want) * 2 ** -10), float(err.max())
