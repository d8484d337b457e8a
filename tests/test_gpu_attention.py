"""GPU parity of the decode attention (oi2_attn_forward through
oi2.GroupedQueryAttention) against the oracle's restatement of
GroupedQueryAttention.forward (engine.py:90-125).

Bar: the attention output (o_proj, fp16) and the new cache rows within max
rel err 1e-2 and cosine >= 0.9999 of the float64 oracle over the same fp8
weights and the same cache contents; cache positions below ``past`` are left
bit for bit; the fused residual is exactly fp16(x + out).
"""
import ctypes

import numpy as np
import pytest
import torch

import oi2
from oi2 import _lib
from oracle import oracle as O
from tests.gpu_helpers import EPS, assert_ffn_close

pytestmark = pytest.mark.gpu
H = 4096
D = 128


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    return torch.device("cuda:0")


def _weights(dev, n_kv, seed, layer=0):
    """A shared-weights dict as splitter.py:175-179 writes it: fp8 e4m3fn
    projections, fp16 input_layernorm."""
    g = torch.Generator(device=dev).manual_seed(seed)
    n_q = H // D

    def w(rows, cols):
        return (torch.randn((rows, cols), generator=g, device=dev) * 0.02).to(torch.float8_e4m3fn)

    p = f"layer_{layer:03d}."
    return {p + "q_proj": w(n_q * D, H), p + "k_proj": w(n_kv * D, H), p + "v_proj": w(n_kv * D, H),
            p + "o_proj": w(H, n_q * D),
            p + "input_layernorm": (1.0 + 0.1 * torch.randn(H, generator=g, device=dev)).half()}


def _cfg(n_kv):
    return {"num_attention_heads": H // D, "num_key_value_heads": n_kv, "hidden_dim": H,
            "rms_norm_eps": EPS}


def _dense(weights, layer=0):
    p = f"layer_{layer:03d}."
    f = lambda n: weights[p + n].float().cpu().numpy().astype(np.float64)
    return (f("q_proj"), f("k_proj"), f("v_proj"), f("o_proj"),
            weights[p + "input_layernorm"].float().cpu().numpy().astype(np.float64))


def _oracle(weights, n_kv, x, cos, sin, cache):
    wq, wk, wv, wo, nw = _dense(weights)
    kv = None if cache is None else (cache[0].float().cpu().numpy(), cache[1].float().cpu().numpy())
    T = x.shape[1]
    return O.gqa_attention(x.float().cpu().numpy(), nw, EPS, wq, wk, wv, wo, H // D, n_kv,
                           cos[:T].cpu().numpy(), sin[:T].cpu().numpy(), kv)


def _check_step(attn, weights, n_kv, x, cos, sin, cache, what):
    """One call against the oracle over the same cache contents; returns the
    call's (out, (k, v))."""
    before = None if cache is None else (cache[0].clone(), cache[1].clone())
    res = torch.empty_like(x)
    out, (k, v) = attn(x, cos, sin, cache, residual_out=res)
    torch.cuda.synchronize()
    ref, (rk, rv) = _oracle(weights, n_kv, x, cos, sin, before)
    print(f"[attn] {what}: out {tuple(out.shape)}, cache {tuple(k.shape)}", flush=True)
    assert_ffn_close(out.float().cpu().numpy(), ref, what=f"{what} out")
    past = 0 if before is None else before[0].shape[2]
    T = x.shape[1]
    assert k.shape == (x.shape[0], n_kv, past + T, D) and v.shape == k.shape
    assert_ffn_close(k[:, :, past:].float().cpu().numpy(), rk[:, :, past:], what=f"{what} new k")
    assert_ffn_close(v[:, :, past:].float().cpu().numpy(), rv[:, :, past:], what=f"{what} new v")
    if before is not None:
        assert torch.equal(k[:, :, :past], before[0]) and torch.equal(v[:, :, :past], before[1])
    assert torch.equal(res, (x.float() + out.float()).half()), f"{what}: fused residual"
    return out, (k, v)


def _rand_cache(dev, B, n_kv, past, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    k = torch.randn((B, n_kv, past, D), generator=g, device=dev).half()
    v = torch.randn((B, n_kv, past, D), generator=g, device=dev).half()
    return k, v


def _forward(w, n_kv, x, cos, sin, k, v, past, causal, batch):
    """oi2_attn_forward over caches of k's own capacity, through the C ABI."""
    L, p = oi2.load_library(), "layer_000."
    T, dev = x.shape[0] // batch, x.device
    s = _lib.Attn(H // D, n_kv, *(w[p + n].data_ptr() for n in ("q_proj", "k_proj", "v_proj", "o_proj", "input_layernorm")))
    nb = L.oi2_attn_workspace_bytes(batch, T, H // D, n_kv, past)
    ws, out = torch.empty(nb, dtype=torch.uint8, device=dev), torch.empty_like(x)
    _lib.check(L.oi2_attn_forward(x.data_ptr(), batch, T, ctypes.byref(s), EPS, cos.data_ptr(), sin.data_ptr(), k.data_ptr(),
                                  v.data_ptr(), k.shape[2], past, int(causal), out.data_ptr(), None, ws.data_ptr(), nb,
                                  _lib.stream_handle(dev)))
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("B,past,n_kv", [(1, 5, 8), (1, 37, 8), (3, 300, 8), (1, 4095, 8), (3, 1000, 8), (2, 100, 32),
                                         (2, 129, 4), (1, 255, 16), (1, 1023, 8), (2, 1024, 8)])
def test_decode_step_against_oracle(dev, B, past, n_kv):
    """One token per sequence over a cache from elsewhere (copied into the
    layer's buffer): query groups of 1, 2, 4, 8; spans up to 1024 positions
    in one workgroup per query head (1024 itself included), longer ones split
    over the sequence (1025 and 4096 positions)."""
    w = _weights(dev, n_kv, seed=past + n_kv)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(past + 8, D, 10000.0, device=dev)
    g = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn((B, 1, H), generator=g, device=dev).half()
    cache = _rand_cache(dev, B, n_kv, past, seed=past)
    _check_step(attn, w, n_kv, x, cos[past:], sin[past:], cache, f"decode B={B} past={past} n_kv={n_kv}")


@pytest.mark.parametrize("B,T,past,n_kv", [(8, 1, 1024, 8), (1, 1, 8191, 8), (1, 1, 8192, 8), (1, 1, 6400, 8),
                                           (1, 1, 6399, 8), (4, 1, 1280, 16), (2, 1, 1055, 32), (1, 5, 2040, 8),
                                           (8, 1, 2100, 4), (7, 1, 1792, 4), (7, 1, 1791, 4)])
def test_long_spans_in_looping_splits(dev, B, T, past, n_kv):
    """Spans whose 256-position splits number at least 208: the last split of
    one position, of all 256 and of most of them, one split fewer (one-shot
    splits), query groups of 1, 2, 4 and 8; keys that grow along the span.  A
    position hardly weighs here: the test after this one gives each split's own."""
    w = _weights(dev, n_kv, seed=past + n_kv)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(past + T, D, 10000.0, device=dev)
    g = torch.Generator(device=dev).manual_seed(11)
    x = torch.randn((B, T, H), generator=g, device=dev).half()
    k, v = _rand_cache(dev, B, n_kv, past, seed=past)
    k *= torch.linspace(0.1, 2.0, past, device=dev).half()[:, None]
    _check_step(attn, w, n_kv, x, cos[past:], sin[past:], (k, v), f"B={B} T={T} past={past} n_kv={n_kv}")


def _row_err(y, ref):
    """Largest error of each row (last axis) over the row's largest value."""
    y, ref = np.asarray(y, np.float64), np.asarray(ref, np.float64)
    return np.abs(y - ref).max(-1) / np.abs(ref).max(-1)


@pytest.mark.parametrize("B,T,past,n_kv", [(8, 1, 1024, 8), (1, 1, 8192, 8), (1, 1, 6400, 8), (1, 1, 6399, 8), (4, 1, 1280, 16),
                                           (2, 1, 1055, 32), (1, 5, 2040, 8), (7, 1, 1792, 4), (1, 1, 1500, 8), (1, 1, 900, 8)])
def test_every_split_of_a_long_span_counts(dev, B, T, past, n_kv):
    """Scores that rise by 4 along the span, so that every chunk of every split
    raises the running max, and about one position in each 64 (every offset,
    the ends of the span, the last split's first position) whose v makes up for
    its probability: each adds 1/64 to the output, whose rows are compared one
    by one.  Half the weight of one of them is past the bar, 3 times the fp16
    rounding of the output (2^-11 of the largest value) and as much again for
    the fp32 exponentials and sums; the oracle with the last position, or the
    last split's first, left out shows that the bar sees one."""
    G, n = 32 // n_kv, past + T
    g = torch.Generator(device=dev).manual_seed(past + n_kv)
    p = "layer_000."

    def cols(rows, count, value=1.0):
        w = torch.zeros((rows, H), device=dev)
        w[:, :count] = value * 2.0 ** -9
        return w.to(torch.float8_e4m3fn)
    # x_n = 1: q = 1 and k = 0.36 in every dim, v = +-32; out is the attention itself
    sign = torch.where(torch.rand((n_kv * D, 1), generator=g, device=dev) < 0.5, -1.0, 1.0)
    w = {p + "q_proj": cols(H, 512), p + "k_proj": cols(n_kv * D, 184), p + "v_proj": cols(n_kv * D, 512, 32.0 * sign),
         p + "o_proj": torch.eye(H, device=dev).to(torch.float8_e4m3fn), p + "input_layernorm": torch.ones(H, device=dev).half()}
    cos, sin = torch.ones((T, D // 2), device=dev), torch.zeros((T, D // 2), device=dev)
    x = torch.ones((B, T, H), device=dev).half()
    t = torch.linspace(0.0, 0.35, past, device=dev).half()
    k = t[:, None].expand(B, n_kv, past, D).contiguous()
    prob = torch.softmax(torch.cat([t.double(), torch.full((T,), 184 / 512, device=dev).double()]) * D ** 0.5, 0)
    at = (torch.arange(0, past, 64, device=dev) + 37 * torch.arange(0, (past + 63) // 64, device=dev) % 64).clamp(max=past - 1)
    last = (n - 1) // 256 * 256
    at = torch.cat([at, torch.tensor([0, past - 1, min(last, past - 1)], device=dev)]).unique()
    v = torch.randn((B, n_kv, past, D), generator=g, device=dev)
    v[:, :, at] = torch.where(torch.rand((B, n_kv, at.numel(), D), generator=g, device=dev) < 0.5, -1.0, 1.0) \
        * (1 / 64 / prob[at]).float()[:, None]
    out, (k, v) = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x, cos, sin, (k, v.half()))
    bar = 3 * 2.0 ** -10
    kn, vn = k.double().cpu().numpy(), v.double().cpu().numpy()

    def reference(keep):
        q = np.ones((B, 32, T, D))
        return O.attention_core(q, kn[:, :, keep], vn[:, :, keep], causal=False).transpose(0, 2, 1, 3)
    every = np.arange(n)
    ref = reference(every)
    err = _row_err(out.float().cpu().numpy().reshape(B, T, 32, D), ref)
    print(f"[attn] B={B} T={T} past={past} n_kv={n_kv}: row error {err.max():.1e}, bar {bar:.1e}", flush=True)
    assert err.max() <= bar
    for lost in {n - 1, min(last, past - 1)}:
        assert _row_err(reference(every[every != lost]), ref).min() > 2 * bar


def _weights_out_is_attention(dev, n_kv, seed):
    w = _weights(dev, n_kv, seed)
    w["layer_000.o_proj"] = torch.eye(H, device=dev).to(torch.float8_e4m3fn)
    return w


@pytest.mark.parametrize("T,past,n_kv", [(400, 0, 8), (700, 0, 16), (3, 100, 8), (3, 1100, 8), (9, 60, 8), (70, 100, 8), (130, 1100, 4),
                                         (600, 33, 8)])
def test_causal_rows_see_their_own_position_and_no_later_one(dev, T, past, n_kv):
    """Causal rows at and beside the edges of tiles of rows and positions, each
    against the oracle's attention over exactly the positions up to its own,
    also behind a cache (which the C ABI allows and the engine does not ask
    for); the oracle with one position fewer or more shows that the bar, 5e-3 of
    the row's largest value, tells them apart."""
    w = _weights_out_is_attention(dev, n_kv, seed=111)
    n = past + T
    cos, sin = (t[past:].contiguous() for t in oi2.rope_tables(n, D, 1e6, device=dev))
    x = torch.randn((T, H), generator=torch.Generator(device=dev).manual_seed(112), device=dev).half()
    k, v = (torch.zeros((1, n_kv, n, D), device=dev).half() for _ in range(2))
    if past:
        for t, r in zip((k, v), _rand_cache(dev, 1, n_kv, past, seed=113)):
            t[:, :, :past] = r
    out = _forward(w, n_kv, x, cos, sin, k, v, past, True, 1).float().cpu().numpy().reshape(T, 32, D)
    kn, vn = k.double().cpu().numpy(), v.double().cpu().numpy()
    xn = O.rmsnorm(x.double().cpu().numpy(), w["layer_000.input_layernorm"].double().cpu().numpy(), EPS).astype(np.float16)
    q = (xn.astype(np.float64) @ w["layer_000.q_proj"].double().cpu().numpy().T).astype(np.float16).astype(np.float64)
    q = O.apply_rope(q.reshape(1, T, 32, D).transpose(0, 2, 1, 3), *(t.half().double().cpu().numpy() for t in (cos, sin)))
    q = q.astype(np.float16).astype(np.float64)
    rows = sorted({r for e in (0, 32, 63, 64, 127, 128, 255, 256, 383, 512, T - 1) for r in (e - 1, e, e + 1) if 0 <= r < T})
    for r in rows:
        see = past + r + 1
        one = lambda m: O.attention_core(q[:, :, r:r + 1], kn[:, :, :m], vn[:, :, :m], causal=False)[0, :, 0]
        ref = one(see)
        err = _row_err(out[r], ref).max()
        assert err <= 5e-3, (r, err)
        for m in (see - 1, see + 1):
            if 0 < m <= n:
                assert _row_err(one(m), ref).max() > 1e-2
    print(f"[attn] T={T} past={past} n_kv={n_kv}: {len(rows)} rows", flush=True)


def test_prefill_then_decode_like_the_engine(dev):
    """engine.py:406-442's use: a causal prefill without a cache, then
    decode steps that pass back the cache the previous call returned (the
    in-place append), each checked over the cache it was given; the RoPE
    positions continue from the cache length (engine.py:414-416)."""
    n_kv, B, T = 8, 2, 5
    w = _weights(dev, n_kv, seed=11)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(64, D, 1e6, device=dev)
    g = torch.Generator(device=dev).manual_seed(12)
    x = torch.randn((B, T, H), generator=g, device=dev).half()
    _, kv = _check_step(attn, w, n_kv, x, cos, sin, None, "prefill B=2 T=5")
    ptr = kv[0].data_ptr()
    for step in range(3):
        past = kv[0].shape[2]
        xt = torch.randn((B, 1, H), generator=g, device=dev).half()
        _, kv = _check_step(attn, w, n_kv, xt, cos[past:past + 1], sin[past:past + 1], kv,
                            f"decode step {step}")
        assert kv[0].data_ptr() == ptr, "the returned cache is appended in place"


def test_rows_beyond_one_launch_and_noncausal_chunk(dev):
    """12 query rows (past the five that one GEMV launch takes), causal
    prefill; then a 3-token chunk over a cache, which the reference runs
    non-causally (is_causal is False whenever a cache is given,
    engine.py:121)."""
    n_kv, B = 8, 3
    w = _weights(dev, n_kv, seed=21)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(64, D, 10000.0, device=dev)
    g = torch.Generator(device=dev).manual_seed(22)
    x = torch.randn((B, 4, H), generator=g, device=dev).half()
    _, kv = _check_step(attn, w, n_kv, x, cos, sin, None, "prefill B=3 T=4")
    x2 = torch.randn((B, 3, H), generator=g, device=dev).half()
    _check_step(attn, w, n_kv, x2, cos[4:], sin[4:], kv, "chunk of 3 over a cache")


def test_cache_growth_and_default_norm(dev):
    """A decode past the buffer's room moves the cache to a larger buffer
    with its contents; a weights dict without input_layernorm uses
    nn.RMSNorm's default weight of ones (engine.py:85-88)."""
    n_kv, B = 8, 1
    w = _weights(dev, n_kv, seed=31)
    del w["layer_000.input_layernorm"]
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(300, D, 10000.0, device=dev)
    g = torch.Generator(device=dev).manual_seed(32)
    x = torch.randn((B, 255, H), generator=g, device=dev).half()
    _, kv = attn(x, cos, sin)
    assert attn.capacity == 256
    w["layer_000.input_layernorm"] = torch.ones(H, dtype=torch.float16, device=dev)
    for step in range(2):
        past = kv[0].shape[2]
        xt = torch.randn((B, 1, H), generator=g, device=dev).half()
        _, kv = _check_step(attn, w, n_kv, xt, cos[past:], sin[past:], kv, f"growth step {step}")
    assert attn.capacity == 512 and kv[0].shape[2] == 257


def test_returned_caches_never_change(dev):
    """Tensors a call returned keep their contents whatever later calls do:
    a second sequence (kv_cache=None), a roll-back to an older, shorter view
    of the cache, and the in-place append of the latest view (which writes
    only past the earlier views' ends).  The reference returns fresh
    torch.cat tensors every call (engine.py:105-109)."""
    n_kv, B = 8, 1
    w = _weights(dev, n_kv, seed=41)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(64, D, 10000.0, device=dev)
    g = torch.Generator(device=dev).manual_seed(42)
    x = torch.randn((B, 6, H), generator=g, device=dev).half()
    _, kv_a = attn(x, cos, sin)
    xt = torch.randn((B, 1, H), generator=g, device=dev).half()
    _, kv_a1 = attn(xt, cos[6:], sin[6:], kv_a)          # in place: kv_a is unchanged
    torch.cuda.synchronize()
    snap = [t.clone() for t in (*kv_a, *kv_a1)]
    x2 = torch.randn((B, 9, H), generator=g, device=dev).half()
    _, kv_b = attn(x2, cos, sin)                          # a second sequence
    x3 = torch.randn((B, 1, H), generator=g, device=dev).half()
    _, kv_r = _check_step(attn, w, n_kv, x3, cos[6:], sin[6:], kv_a, "roll back to 6 positions")
    torch.cuda.synchronize()
    for t, s in zip((*kv_a, *kv_a1), snap):
        assert torch.equal(t, s), "a returned cache changed"
    assert kv_b[0].shape[2] == 9 and kv_r[0].shape[2] == 7
    assert kv_b[0].data_ptr() != kv_a[0].data_ptr() and kv_r[0].data_ptr() != kv_a[0].data_ptr()
    # the roll-back's new position differs from the first sequence's own 7th
    assert not torch.equal(kv_r[0][:, :, 6], kv_a1[0][:, :, 6])


def test_rewind_decodes_a_position_again_in_place(dev):
    """rewind(n) is the one opt-in roll-back that reuses the buffer: a view
    of length n then appends in place at position n, the first n positions
    stay bit for bit, and decoding the same token at the same position twice
    gives the same output and cache row (the oracle checks the step)."""
    n_kv, B = 8, 1
    w = _weights(dev, n_kv, seed=43)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(64, D, 10000.0, device=dev)
    g = torch.Generator(device=dev).manual_seed(44)
    x = torch.randn((B, 10, H), generator=g, device=dev).half()
    _, kv = attn(x, cos, sin)
    view = (kv[0][:, :, :10], kv[1][:, :, :10])
    head = [t.clone() for t in view]
    xt = torch.randn((B, 1, H), generator=g, device=dev).half()
    out1, kv1 = _check_step(attn, w, n_kv, xt, cos[10:], sin[10:], view, "decode at 10")
    row1 = (kv1[0][:, :, 10].clone(), kv1[1][:, :, 10].clone())
    attn.rewind(10)
    out2, kv2 = attn(xt, cos[10:], sin[10:], view)
    torch.cuda.synchronize()
    assert kv2[0].data_ptr() == kv[0].data_ptr(), "rewind must reuse the layer's buffer"
    assert torch.equal(out1, out2)
    assert torch.equal(kv2[0][:, :, 10], row1[0]) and torch.equal(kv2[1][:, :, 10], row1[1])
    for t, s in zip(view, head):
        assert torch.equal(t, s)
    with pytest.raises(ValueError):
        attn.rewind(12)


@pytest.mark.parametrize("B,T,n_kv", [(1, 9, 8), (1, 63, 32), (1, 64, 8), (2, 65, 4), (1, 129, 8), (3, 43, 16),
                                      (1, 400, 8), (1, 700, 32), (11, 1, 8), (6, 1, 4), (1, 16, 32), (1, 17, 8),
                                      (2, 16, 16), (1, 33, 8), (1, 17, 32)])
def test_prompt_rows_on_the_matrix_cores(dev, B, T, n_kv):
    """Rows at the edges of the projections' kernels for a few rows (6 to 16, 17
    to 32), of the prompt projections' 64- and 128-row tiles and
    of their choice of tile (400 rows with 48 heads and 700 rows with 96 fill
    more than one tile per CU), several sequences with rows of each in one
    tile, a batch of single rows over a cache."""
    w = _weights(dev, n_kv, seed=51 + T)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    past = 33 if T == 1 else 0
    cos, sin = oi2.rope_tables(past + T, D, 1e6, device=dev)
    x = torch.randn((B, T, H), generator=torch.Generator(device=dev).manual_seed(52), device=dev).half()
    cache = _rand_cache(dev, B, n_kv, past, seed=53) if past else None
    _check_step(attn, w, n_kv, x, cos[past:], sin[past:], cache, f"prompt B={B} T={T} n_kv={n_kv}")


@pytest.mark.parametrize("B,T,past,n_kv", [(1, 9, 70, 8), (2, 64, 64, 32), (1, 65, 1023, 8), (2, 33, 4000, 4),
                                           (1, 128, 0, 16), (1, 1100, 0, 8)])
def test_prompt_attention_on_the_matrix_cores(dev, B, T, past, n_kv):
    """Query rows at the edges of the prompt attention's 64-row tiles against
    spans at the edges of its 64-position ones: chunks over a cache (every row
    sees every position) and causal prompts, query groups of 1, 2, 4 and 8,
    several sequences."""
    w = _weights(dev, n_kv, seed=61 + T)
    attn = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))
    cos, sin = oi2.rope_tables(past + T, D, 1e6, device=dev)
    x = torch.randn((B, T, H), generator=torch.Generator(device=dev).manual_seed(62), device=dev).half()
    cache = _rand_cache(dev, B, n_kv, past, seed=63) if past else None
    _check_step(attn, w, n_kv, x, cos[past:], sin[past:], cache, f"attention B={B} T={T} past={past} n_kv={n_kv}")


@pytest.mark.parametrize("bad", [5, 40, 63, 64, 90])
def test_a_prompt_row_does_not_see_later_non_finite_values(dev, bad):
    """A position whose v overflows fp16 (and so is inf) spoils the rows that
    see it and no earlier row, wherever it lies in a tile of positions: the
    rows before it equal those of the prompt cut off before it."""
    n_kv, T = 8, 100
    w = _weights(dev, n_kv, seed=71)
    w["layer_000.v_proj"] = torch.full((n_kv * D, H), 96.0, device=dev).to(torch.float8_e4m3fn)
    w["layer_000.input_layernorm"] = torch.ones(H, dtype=torch.float16, device=dev)
    cos, sin = oi2.rope_tables(T, D, 1e6, device=dev)
    x = torch.randn((1, T, H), generator=torch.Generator(device=dev).manual_seed(72), device=dev).half()
    x[0, bad] = 1.0                                        # v = 4096 * 96
    out, (_, v) = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x, cos, sin)
    cut, _ = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x[:, :bad].contiguous(), cos, sin)
    assert torch.isinf(v[0, :, bad]).all() and torch.isfinite(v[0, :, :bad]).all()
    assert torch.isfinite(out[0, :bad]).all()
    assert_ffn_close(out[0, :bad].float().cpu().numpy(), cut[0].float().cpu().numpy(), tol=2e-3, what="rows before")
    assert not torch.isfinite(out[0, bad:]).any()


def _infinite_setup(dev, n_kv):
    """Weights with which a token of ones has v = 4096 * 24, infinite in fp16,
    in every dim, and every output is the sum of the attention's dims: rows
    that see the token come out as inf, not NaN."""
    w = _weights(dev, n_kv, seed=91)
    w["layer_000.v_proj"] = torch.full((n_kv * D, H), 24.0, device=dev).to(torch.float8_e4m3fn)
    w["layer_000.o_proj"] = torch.full((H, H), 2.0 ** -9, device=dev).to(torch.float8_e4m3fn)
    w["layer_000.input_layernorm"] = torch.ones(H, dtype=torch.float16, device=dev)
    return w


@pytest.mark.parametrize("T,bad", [(100, 40), (200, 5), (200, 130), (600, 5), (600, 300), (600, 599)])
def test_prompt_rows_that_see_an_infinite_value_are_infinite(dev, T, bad):
    """Tiles of positions that some row of a workgroup does not see, and tiles that every row
    of a workgroup sees (where an infinite v times the zero low part of its
    probability must not become NaN), with four position parts a workgroup
    (up to 512 rows) and with two."""
    n_kv = 8
    w = _infinite_setup(dev, n_kv)
    cos, sin = oi2.rope_tables(T, D, 1e6, device=dev)
    x = torch.randn((1, T, H), generator=torch.Generator(device=dev).manual_seed(92), device=dev).half()
    x[0, bad] = 1.0
    out, (_, v) = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x, cos, sin)
    cut, _ = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x[:, :bad].contiguous(), cos, sin)
    assert torch.isposinf(v[0, :, bad]).all() and torch.isfinite(v[0, :, :bad]).all()
    assert torch.isposinf(out[0, bad:]).all()
    assert_ffn_close(out[0, :bad].float().cpu().numpy(), cut[0].float().cpu().numpy(), tol=2e-3, what="rows before")


@pytest.mark.parametrize("T,past,at,value", [(16, 300, 7, "inf"), (70, 300, 290, "-inf"), (600, 200, 130, "inf"),
                                             (16, 300, 100, "nan")])
def test_rows_over_a_cache_with_a_non_finite_value(dev, T, past, at, value):
    """A chunk over a cache (every row sees every position) one of whose v is
    not finite: every output is that value."""
    n_kv = 8
    w = _infinite_setup(dev, n_kv)
    cos, sin = oi2.rope_tables(past + T, D, 1e6, device=dev)
    x = torch.randn((1, T, H), generator=torch.Generator(device=dev).manual_seed(93), device=dev).half()
    k, v = _rand_cache(dev, 1, n_kv, past, seed=94)
    v[0, :, at] = float(value)
    out, _ = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x, cos[past:], sin[past:], (k, v))
    want = torch.full_like(out, float(value))
    assert torch.equal(torch.nan_to_num(out, nan=1.0, posinf=2.0, neginf=3.0),
                       torch.nan_to_num(want, nan=1.0, posinf=2.0, neginf=3.0))


@pytest.mark.parametrize("past", [300, 1500, 1535, 6399, 6400, 6655])
def test_a_decoded_token_with_an_infinite_value(dev, past):
    """One token whose own v is infinite, at every place of the last split
    (short spans, one-shot and looping splits): the output is infinite.  The
    loads past the span must not meet that v with a probability of 0."""
    n_kv = 8
    w = _infinite_setup(dev, n_kv)
    cos, sin = oi2.rope_tables(past + 1, D, 1e6, device=dev)
    x = torch.ones((1, 1, H), device=dev).half()
    out, _ = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x, cos[past:], sin[past:], _rand_cache(dev, 1, n_kv, past, seed=95))
    assert torch.isposinf(out).all()


@pytest.mark.parametrize("rows", [6, 17, 33, 400, 700])
def test_a_token_gets_the_same_k_and_v_whichever_projection_runs(dev, rows):
    """The cached k and v of five tokens from a call of their own and from one
    with more rows (each of the projections' kernels and tile sizes): RoPE
    rounds alike in all of them, so that only the order of the fp32 sums
    differs.  Over 4096 products that is up to 3e-7 of the result's rms
    (simulated with 8 to 512 chains), which moves 0.3 % of the fp16 values; a
    RoPE rounded in another place moves 22 % of k's."""
    n_kv, n, at = 8, 5, 1000
    w = _weights(dev, n_kv, seed=81)
    cos, sin = oi2.rope_tables(at + rows, D, 1e6, device=dev)
    x = torch.randn((1, rows, H), generator=torch.Generator(device=dev).manual_seed(82), device=dev).half()
    few = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x[:, :n].contiguous(), cos[at:], sin[at:])[1]
    many = oi2.GroupedQueryAttention(0, w, _cfg(n_kv))(x, cos[at:], sin[at:])[1]
    for name, a, b in zip("kv", few, many):
        share = float((a != b[:, :, :n]).float().mean())
        print(f"[attn] {rows} rows: {share:.2%} of {name} differ from the call of {n}", flush=True)
        assert share <= 0.02, name


def test_more_rows_than_one_projection_launch_addresses(dev):
    """262146 sequences of one token, past the rows that one launch's 32-bit
    offsets reach (a multiple of 128 below 2^31 / 8192): the last 130 rows equal
    those of a call of their own, but for the order of the fp32 sums."""
    n_kv, B, n = 4, 262016 + 130, 130
    w = _weights(dev, n_kv, seed=101)
    cos, sin = (t[7:].contiguous() for t in oi2.rope_tables(8, D, 1e6, device=dev))
    x = torch.randn((B, H), generator=torch.Generator(device=dev).manual_seed(102), device=dev, dtype=torch.float16)
    res = []
    for rows in (x, x[-n:].contiguous(), x[:n].contiguous()):
        k, v = (torch.full((rows.shape[0], n_kv, 1, D), 9.0, device=dev, dtype=torch.float16) for _ in range(2))
        res.append((_forward(w, n_kv, rows, cos, sin, k, v, 0, True, rows.shape[0]), k, v))
    for what, part, alone in (("last", slice(-n, None), res[1]), ("first", slice(0, n), res[2])):
        for a, b in zip(res[0], alone):
            assert_ffn_close(a[part].float().cpu().numpy(), b.float().cpu().numpy(), tol=2e-3, what=f"{what} rows")
