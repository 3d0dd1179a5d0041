"""GPU parity of the layer input stage (run_layer: RMSNorm, QKV projection, RoPE) and of run_layer.

Bars (the stage specification is in oracle/layer_oracle.py):
* projection: every output element within one bf16 ulp of the float64 product plus the fp32
  accumulation term 2^-20 * sum |x w|;
* RMSNorm, read through an identity projection: every element within one bf16 ulp of the
  float64 value, and at least 99 % equal to its nearest-even rounding;
* RoPE: word for word equal to the fp32 restatement applied to the GPU's own unrotated
  projection (same bf16 inputs, same operations);
* run_layer: within 2 bf16 ulp per row of the float64 attention of the GPU's Q/K/V, K/V
  rows in the cache identical to the device-pointer stage's, and within 3 ulp of the float64
  chain (rounding to bf16 at the same points); with KV260 numerics, word for word equal to
  the C restatement of the board arithmetic on the GPU's Q/K/V.
"""
import ctypes

import numpy as np
import pytest

from lara_amd import _lib
from lara_amd.attn_driver import AttentionAccelerator
from oracle import gqa_oracle as orc
from oracle import layer_oracle as lo
from tests._gen import bf16_normal

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(words: np.ndarray):
    return torch.from_numpy(np.ascontiguousarray(words).view(np.int16)).cuda()


def host(t) -> np.ndarray:
    return t.cpu().numpy().view(np.uint16)


def stage(acc, x, wq, wk, wv, gamma, *, b=0, q_pos_base=0, kv_pos_base=0, row0=0, rope=True, eps=1e-5,
          fused=False):
    """Run gqa_layer_qkv_device; returns Q [H_q, L, D] and the K/V rows written.  fused=True
    stores Wq, Wk, Wv back to back (the library then runs one projection GEMM)."""
    L, hidden = x.shape
    if fused:
        wqkv = dev(np.concatenate([wq, wk, wv]))
        nq, nkv = wq.shape[0], wk.shape[0]
        bufs = [dev(x), wqkv[:nq], wqkv[nq:nq + nkv], wqkv[nq + nkv:]]
    else:
        bufs = [dev(a) for a in (x, wq, wk, wv)]
    g = dev(gamma) if gamma is not None else None
    q = torch.empty((acc.n_q_heads, L, acc.head_dim), dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()  # the uploads ran on torch's stream; the stage runs on the engine's
    acc.layer_qkv_device(bufs[0].data_ptr(), L, hidden, bufs[1].data_ptr(), bufs[2].data_ptr(), bufs[3].data_ptr(),
                         g.data_ptr() if g is not None else None, q.data_ptr(), b=b, q_pos_base=q_pos_base,
                         kv_pos_base=kv_pos_base, kv_row0=row0, rope=rope, rms_eps=eps)
    torch.cuda.synchronize()
    k, v = acc.read_kv(b, row0, L)
    return host(q), k, v


def weights(rng, nq, nkv, hidden):
    s = 1.0 / np.sqrt(hidden)
    return bf16_normal(rng, (nq, hidden), s), bf16_normal(rng, (nkv, hidden), s), bf16_normal(rng, (nkv, hidden), s)


@pytest.mark.parametrize("fused", [False, True])
def test_first_call_of_a_shape_equals_the_tuned_calls(fused):
    # The first call of a projection shape times hipBLASLt's candidates (running each on the
    # destination) and keeps the fastest; that call and the later ones (cached pick, no timing)
    # must leave the same words, and a new shape in between must not disturb the cached plan.
    print(f"[layer] tuned projection repeatability fused={fused}", flush=True)
    rng = np.random.default_rng(77)
    with AttentionAccelerator(n_q_heads=8, n_kv_heads=2, head_dim=128, max_seq_len=384) as acc:
        x = bf16_normal(rng, (192, 2048))
        wq, wk, wv = weights(rng, 1024, 256, 2048)
        gamma = orc.fp32_to_bf16_u16(1 + 0.1 * rng.standard_normal(2048, dtype=np.float32))
        first = stage(acc, x, wq, wk, wv, gamma, row0=5, fused=fused)
        other = stage(acc, x[:64], wq, wk, wv, gamma, row0=200, fused=fused)  # another shape
        second = stage(acc, x, wq, wk, wv, gamma, row0=5, fused=fused)
        third = stage(acc, x, wq, wk, wv, gamma, row0=5, fused=fused)
    assert other[0].shape[1] == 64
    for a, b, c in zip(first, second, third):
        assert np.array_equal(a, b) and np.array_equal(b, c)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("hidden,L", [(768, 37), (1001, 5), (4096, 64)])
def test_projection_within_fp32_accumulation_bound(hidden, L, fused):
    print(f"[layer] projection hidden={hidden} L={L} fused={fused}", flush=True)
    rng = np.random.default_rng(hidden + L)
    with AttentionAccelerator(n_q_heads=8, n_kv_heads=2, head_dim=128, max_seq_len=128) as acc:
        x = bf16_normal(rng, (L, hidden))
        wq, wk, wv = weights(rng, 1024, 256, hidden)
        q, k, v = stage(acc, x, wq, wk, wv, None, rope=False, row0=3, fused=fused)
    for got_heads, w, H in ((q, wq, 8), (k, wk, 2), (v, wv, 2)):
        got = orc.bf16_u16_to_fp32(got_heads).astype(np.float64).transpose(1, 0, 2).reshape(L, H * 128)
        exact = lo.project_exact(x, w)
        bound = lo.projection_error_bound(x, w)
        assert np.all(np.abs(got - exact) <= bound), float(np.max(np.abs(got - exact) / bound))
        same = np.mean(orc.bf16_rne(exact.astype(np.float32)) == orc.fp32_to_bf16_u16(got.astype(np.float32)))
        assert same > 0.95


@pytest.mark.parametrize("extra_cols", [0, 3, 8192])
def test_rms_norm_through_identity_projection(extra_cols):
    """Wq = [I | 0] makes Q the first H_q*D columns of the normalised x exactly (fp32 sums of
    one non-zero product); extra_cols = 3 exercises the unaligned (scalar) kernel path and
    8192 rows longer than the register-cached part."""
    nq = 1024
    hidden = nq + extra_cols
    L = 19
    print(f"[layer] rms_norm hidden={hidden}", flush=True)
    rng = np.random.default_rng(50 + extra_cols)
    x = bf16_normal(rng, (L, hidden), 2.0)
    x[3] = orc.fp32_to_bf16_u16(np.full(hidden, 0.001, np.float32))  # a small row: eps matters
    gamma = orc.fp32_to_bf16_u16((1.0 + 0.2 * rng.standard_normal(hidden)).astype(np.float32))
    wq = np.zeros((nq, hidden), np.uint16)
    wq[np.arange(nq), np.arange(nq)] = 0x3F80  # 1.0
    _, wk, wv = weights(rng, nq, 256, hidden)
    with AttentionAccelerator(n_q_heads=8, n_kv_heads=2, head_dim=128, max_seq_len=64) as acc:
        q, _, _ = stage(acc, x, wq, wk, wv, gamma, rope=False, eps=1e-5)
    got = orc.bf16_u16_to_fp32(q).astype(np.float64).transpose(1, 0, 2).reshape(L, nq)
    exact = lo.rms_norm_exact(x, gamma, 1e-5)[:, :nq]
    assert np.all(np.abs(got - exact) <= orc.bf16_ulp(exact))
    assert np.mean(orc.bf16_rne(exact.astype(np.float32)) == orc.fp32_to_bf16_u16(got.astype(np.float32))) > 0.99


@pytest.mark.parametrize("qb,kb", [(0, 0), (5, 2), (60000, 59990)])
def test_rope_is_word_exact(qb, kb):
    print(f"[layer] rope q_pos_base={qb} kv_pos_base={kb}", flush=True)
    rng = np.random.default_rng(qb + 7)
    L, hidden = 40, 512
    x = bf16_normal(rng, (L, hidden))
    gamma = orc.fp32_to_bf16_u16((1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32))
    wq, wk, wv = weights(rng, 1024, 256, hidden)
    with AttentionAccelerator(n_q_heads=8, n_kv_heads=2, head_dim=128, max_seq_len=64) as acc:
        q0, k0, v0 = stage(acc, x, wq, wk, wv, gamma, rope=False, q_pos_base=qb, kv_pos_base=kb)
        q1, k1, v1 = stage(acc, x, wq, wk, wv, gamma, rope=True, q_pos_base=qb, kv_pos_base=kb)
    assert np.array_equal(q1, lo.apply_rope(q0, qb))
    assert np.array_equal(k1, lo.apply_rope(k0, kb))
    assert np.array_equal(v1, v0)
    if qb == 0:
        assert np.array_equal(q1[:, 0], q0[:, 0])  # position 0 is not rotated


def test_rope_head_dim_64():
    rng = np.random.default_rng(64)
    L, hidden = 9, 256
    x = bf16_normal(rng, (L, hidden))
    wq, wk, wv = weights(rng, 8 * 64, 2 * 64, hidden)
    with AttentionAccelerator(n_q_heads=8, n_kv_heads=2, head_dim=64, max_seq_len=32) as acc:
        q0, k0, _ = stage(acc, x, wq, wk, wv, None, rope=False, q_pos_base=11, kv_pos_base=4)
        q1, k1, _ = stage(acc, x, wq, wk, wv, None, rope=True, q_pos_base=11, kv_pos_base=4)
    assert np.array_equal(q1, lo.apply_rope(q0, 11)) and np.array_equal(k1, lo.apply_rope(k0, 4))


def _layer_inputs(rng, L, hidden=4096):
    x = bf16_normal(rng, (L, hidden))
    wq, wk, wv = weights(rng, 4096, 1024, hidden)
    gamma = orc.fp32_to_bf16_u16((1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32))
    return x, wq, wk, wv, gamma


@pytest.mark.parametrize("L,causal,qb,kb", [(64, True, 0, 0), (100, True, 7, 7), (33, False, 3, 0)])
def test_run_layer_llama3_shape(L, causal, qb, kb):
    print(f"[layer] run_layer L={L} causal={causal} qb={qb} kb={kb}", flush=True)
    rng = np.random.default_rng(L * 3 + qb)
    x, wq, wk, wv, gamma = _layer_inputs(rng, L)
    with AttentionAccelerator(batch=2) as acc:
        out = acc.run_layer(x, wq, wk, wv, gamma, q_pos_base=qb, kv_pos_base=kb, causal=causal)
        prof = acc.last_profile.to_dict()
        k_layer, v_layer = acc.read_kv(0, 0, L)
        q, k, v = stage(acc, x, wq, wk, wv, gamma, b=1, q_pos_base=qb, kv_pos_base=kb, fused=True)
    assert out.dtype == np.float32 and out.shape == (L, 4096)
    assert prof["host_qkv_projection_ms"] > 0 and prof["host_rope_ms"] > 0 and prof["layer_total_ms"] > 0
    assert np.array_equal(k_layer, k) and np.array_equal(v_layer, v)
    words = orc.fp32_to_bf16_u16(out.reshape(L, 32, 128).transpose(1, 0, 2))
    ref, _ = orc.attention(orc.bf16_u16_to_fp32(q), orc.bf16_u16_to_fp32(k), orc.bf16_u16_to_fp32(v),
                           causal=causal, q_pos_base=qb, kv_pos_base=kb)
    assert float(orc.row_ulp_error(words, ref).max()) <= 2.0
    # the float64 chain, rounded to bf16 at the stage boundaries of the specification
    y = orc.bf16_rne(lo.rms_norm_exact(x, gamma, 1e-5).astype(np.float32))
    proj = [orc.bf16_rne(lo.project_exact(y, w).astype(np.float32)) for w in (wq, wk, wv)]
    qc = lo.apply_rope(lo.reshape_to_heads(proj[0], 32, 128), qb)
    kc = lo.apply_rope(lo.reshape_to_heads(proj[1], 8, 128), kb)
    vc = lo.reshape_to_heads(proj[2], 8, 128)
    chain, _ = orc.attention(orc.bf16_u16_to_fp32(qc), orc.bf16_u16_to_fp32(kc), orc.bf16_u16_to_fp32(vc),
                             causal=causal, q_pos_base=qb, kv_pos_base=kb)
    assert float(orc.row_ulp_error(words, chain).max()) <= 3.0


def test_run_layer_kv260_numerics_is_word_exact():
    from oracle import rtl_exact as rtl

    rng = np.random.default_rng(260)
    L = 48
    x, wq, wk, wv, gamma = _layer_inputs(rng, L)
    with AttentionAccelerator(batch=2, numerics="kv260") as acc:
        out = acc.run_layer(x, wq, wk, wv, gamma, q_pos_base=2, kv_pos_base=2, causal=True)
        q, k, v = stage(acc, x, wq, wk, wv, gamma, b=1, q_pos_base=2, kv_pos_base=2, fused=True)
    want, _, _ = rtl.attention(q, k, v, causal=True, q_pos_base=2, kv_pos_base=2)
    got = orc.fp32_to_bf16_u16(out.reshape(L, 32, 128).transpose(1, 0, 2))
    assert np.array_equal(got, want)


def test_run_layer_rejects_bad_shapes():
    rng = np.random.default_rng(1)
    x, wq, wk, wv, gamma = _layer_inputs(rng, 8, hidden=256)
    with AttentionAccelerator() as acc:
        with pytest.raises(ValueError):
            acc.run_layer(x, wq[:, :100], wk, wv)
        with pytest.raises(ValueError):
            acc.run_layer(x, wq, wk, wv, gamma[:10])
        with pytest.raises(ValueError):
            acc.run_layer(x[None], wq, wk, wv)
        with pytest.raises(ValueError):
            acc.run_layer(bf16_normal(rng, (513, 256)), wq, wk, wv)  # beyond max_seq_len
        with pytest.raises(ValueError):
            acc.run_layer(x, wq, wk, wv, rms_eps=float("nan"))
        out = acc.run_layer(x, wq, wk, wv, gamma, rope=False)
        assert out.shape == (8, 4096) and np.isfinite(out).all()


def test_layer_at_2048_tokens_sampled_rows():
    """The Llama-3-8B layer at 2048 tokens (hidden 4096, 32q/8kv, D 128): RMSNorm, the fused QKV
    projection and RoPE over every row, then one causal prefill launch over them (paired row blocks);
    rows at the start, middle and end of every head against the float64 chain rounded to bf16 at the
    stage boundaries, within 3 bf16 ulp as for run_layer."""
    rng = np.random.default_rng(2048)
    L = 2048
    x, wq, wk, wv, gamma = _layer_inputs(rng, L)
    with AttentionAccelerator(max_seq_len=L, max_q_len=L) as acc:
        print("[layer] 2048-token stage", flush=True)
        q, k, v = stage(acc, x, wq, wk, wv, gamma, fused=True)
        print("[layer] 2048-token causal attention", flush=True)
        out = acc.prefill_chunk(q, q_pos_base=0, kv_len=L, causal=True)
        assert acc.last_prefill_plan() == ("paired", 1)
    y = orc.bf16_rne(lo.rms_norm_exact(x, gamma, 1e-5).astype(np.float32))
    kc = lo.apply_rope(lo.reshape_to_heads(orc.bf16_rne(lo.project_exact(y, wk).astype(np.float32)), 8, 128), 0)
    vc = lo.reshape_to_heads(orc.bf16_rne(lo.project_exact(y, wv).astype(np.float32)), 8, 128)
    for r0 in (0, 992, 1984):  # 64 rows each
        qc = lo.apply_rope(
            lo.reshape_to_heads(orc.bf16_rne(lo.project_exact(y[r0:r0 + 64], wq).astype(np.float32)), 32, 128), r0)
        chain, _ = orc.attention(orc.bf16_u16_to_fp32(qc), orc.bf16_u16_to_fp32(kc[:, :r0 + 64]),
                                 orc.bf16_u16_to_fp32(vc[:, :r0 + 64]), causal=True, q_pos_base=r0)
        assert float(orc.row_ulp_error(out[:, r0:r0 + 64], chain).max()) <= 3.0, r0


def assert_same_stage(a, b):
    """Two stages whose products may be summed in different orders (the library's algorithm is each context's own
    choice): a product near a rounding boundary goes one bf16 ulp either way, and RoPE carries both of a pair's
    into each, rounding again."""
    a, b = (orc.bf16_u16_to_fp32(t).astype(np.float64) for t in (a, b))
    pair = np.maximum(np.hypot(b[..., 0::2], b[..., 1::2]), 2.0 ** -6).repeat(2, axis=-1).astype(np.float32)
    assert np.all(np.abs(a - b) <= 3 * orc.bf16_ulp(pair))


@pytest.mark.parametrize("hidden,L,hq,hkv,d", [(1024, 1, 8, 2, 128), (1024, 16, 8, 2, 64), (2048, 3, 16, 8, 128),
                                               (4096, 1, 32, 8, 128), (4096, 15, 32, 8, 128), (4096, 16, 32, 2, 64),
                                               (4096, 17, 32, 8, 128), (8192, 1, 64, 8, 128), (8192, 8, 64, 8, 128),
                                               (8192, 9, 8, 2, 128), (4096, 5, 1, 1, 64)])
def test_few_tokens_stage(hidden, L, hq, hkv, d):
    """The one-launch stage (up to 16 tokens, 8 at hidden 8192; the others take the general one): the projection
    within its fp32 bound, RMSNorm through it, RoPE word for word, and the same words from separate weights and on
    a paged cache (the general stage: up to the order of its sums)."""
    print(f"[layer] few tokens hidden={hidden} L={L} hq={hq} hkv={hkv} d={d}", flush=True)
    rng = np.random.default_rng(hidden + L + d)
    x = bf16_normal(rng, (L, hidden), 3.0)
    wq, wk, wv = weights(rng, hq * d, hkv * d, hidden)
    gamma = orc.fp32_to_bf16_u16((1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32))
    kw = dict(n_q_heads=hq, n_kv_heads=hkv, head_dim=d, max_seq_len=128)
    with AttentionAccelerator(**kw) as acc:
        plain = stage(acc, x, wq, wk, wv, None, rope=False, row0=3)
        fused = stage(acc, x, wq, wk, wv, None, rope=False, row0=3, fused=True)
        normed = stage(acc, x, wq, wk, wv, gamma, rope=False, row0=60)
        roped = stage(acc, x, wq, wk, wv, gamma, row0=60, q_pos_base=70001, kv_pos_base=60)
    with AttentionAccelerator(page_size=64, n_pages=3, **kw) as acc:
        acc.reserve(0, 128)
        paged = stage(acc, x, wq, wk, wv, gamma, row0=60, q_pos_base=70001, kv_pos_base=60)
    y = orc.bf16_rne(lo.rms_norm_exact(x, gamma, 1e-5).astype(np.float32))
    for got_heads, xin in ((plain, x), (normed, y)):
        for g, w, H in zip(got_heads, (wq, wk, wv), (hq, hkv, hkv)):
            got = orc.bf16_u16_to_fp32(g).astype(np.float64).transpose(1, 0, 2).reshape(L, H * d)
            bound = lo.projection_error_bound(xin, w)
            if xin is y:  # a row's y may round the other way where fp32 sums differ from float64's: one bf16 ulp of 1 % of it
                flips = np.abs(orc.bf16_u16_to_fp32(y).astype(np.float64)) * 2.0 ** -8
                bound = bound + 5.0 * np.sqrt(0.01 * (flips ** 2) @ (orc.bf16_u16_to_fp32(w).astype(np.float64).T ** 2))
            err = np.abs(got - lo.project_exact(xin, w))
            assert np.all(err <= bound), float(np.max(err / bound))
    for a, b, c, e in zip(plain, fused, roped, paged):
        if L <= (8 if hidden > 4096 else 16):
            assert np.array_equal(a, b) and np.array_equal(c, e)
        else:
            assert_same_stage(a, b)
            assert_same_stage(c, e)
    assert np.array_equal(roped[0], lo.apply_rope(normed[0], 70001))
    assert np.array_equal(roped[1], lo.apply_rope(normed[1], 60)) and np.array_equal(roped[2], normed[2])


def test_few_tokens_stage_keeps_the_general_calls():
    """What the one-launch stage does not take still runs: x off 16-byte alignment, and Q written over x."""
    rng = np.random.default_rng(31)
    L, hidden = 4, 1024
    x = bf16_normal(rng, (L, hidden))
    wq, wk, wv = weights(rng, 1024, 256, hidden)
    gamma = orc.fp32_to_bf16_u16((1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32))
    with AttentionAccelerator(n_q_heads=8, n_kv_heads=2, head_dim=128, max_seq_len=64) as acc:
        want = stage(acc, x, wq, wk, wv, gamma)
        bufs = [dev(a) for a in (wq, wk, wv, gamma)]
        shifted = torch.empty(L * hidden + 1, dtype=torch.int16, device="cuda")
        shifted[1:] = dev(x).reshape(-1)
        q = torch.empty((8, L, 128), dtype=torch.int16, device="cuda")
        over = dev(x).clone()  # [4][1024] words: Q's [8][4][128] lands on them
        for src, dst in ((shifted[1:], q), (over, over)):
            print(f"[layer] general call src % 16 = {src.data_ptr() % 16} over={dst is over}", flush=True)
            torch.cuda.synchronize()
            acc.layer_qkv_device(src.data_ptr(), L, hidden, *(t.data_ptr() for t in bufs), dst.data_ptr())
            torch.cuda.synchronize()
            got = host(dst).reshape(8, L, 128)
            assert_same_stage(got, want[0])


def _stage_launches(acc):
    """Launches of the stages since profiling was switched on: (RMSNorm, projection, RoPE)."""
    counts = (ctypes.c_int32 * _lib.GQA_TIMER_COUNT)()
    _lib.check(acc._lib.gqa_kernel_launch_counts(acc._ctx, counts, _lib.GQA_TIMER_COUNT), "counts")
    return tuple(int(counts[t]) for t in (_lib.GQA_TIMER_NORM, _lib.GQA_TIMER_PROJECTION, _lib.GQA_TIMER_ROPE))


@pytest.mark.parametrize("hidden,L,hq,hkv,d,one", [(1024, 16, 8, 2, 64, True), (2048, 3, 16, 8, 128, True),
                                                   (4096, 16, 32, 8, 128, True), (4096, 17, 32, 8, 128, False),
                                                   (8192, 8, 64, 8, 128, True), (8192, 9, 8, 2, 128, False),
                                                   (3072, 4, 8, 2, 128, False)])
def test_few_tokens_stage_is_one_launch(hidden, L, hq, hkv, d, one):
    """Up to 16 tokens (8 at hidden 8192) of a hidden size that has one take one launch, timed as the projection;
    the others RMSNorm, the library's product and RoPE."""
    print(f"[layer] launches hidden={hidden} L={L} hq={hq} hkv={hkv}", flush=True)
    rng = np.random.default_rng(hidden + L)
    wq, wk, wv = weights(rng, hq * d, hkv * d, hidden)
    gamma = orc.fp32_to_bf16_u16(np.ones(hidden, np.float32))
    with AttentionAccelerator(n_q_heads=hq, n_kv_heads=hkv, head_dim=d, max_seq_len=64) as acc:
        _lib.check(acc._lib.gqa_set_option(acc._ctx, _lib.GQA_OPT_PROFILE, 1), "profile")
        stage(acc, bf16_normal(rng, (L, hidden)), wq, wk, wv, gamma)
        assert _stage_launches(acc) == ((0, 1, 0) if one else (1, 1, 1))


@pytest.mark.parametrize("hidden,L,hq,hkv", [(4096, 2, 64, 8), (1024, 3, 128, 16), (2048, 1, 100, 50),
                                             (1024, 16, 128, 64), (8192, 2, 128, 16)])
def test_few_tokens_stage_of_many_tiles(hidden, L, hq, hkv):
    """Work-groups of 2 to 8 output tiles in turn (on 256 CUs: 640, 1280, 1600 and 2048 tiles of 16 rows; 8192: two
    chunks of the product each), odd counts of chunks among them: every projected row within its fp32 bound, RoPE
    word for word, in one launch."""
    d = 128
    print(f"[layer] many tiles hidden={hidden} L={L} hq={hq} hkv={hkv}", flush=True)
    rng = np.random.default_rng(hidden + hq + L)
    x = bf16_normal(rng, (L, hidden))
    wq, wk, wv = weights(rng, hq * d, hkv * d, hidden)
    with AttentionAccelerator(n_q_heads=hq, n_kv_heads=hkv, head_dim=d, max_seq_len=64) as acc:
        _lib.check(acc._lib.gqa_set_option(acc._ctx, _lib.GQA_OPT_PROFILE, 1), "profile")
        plain = stage(acc, x, wq, wk, wv, None, rope=False, row0=3)
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert _stage_launches(acc) == (0, 1, 0)
        roped = stage(acc, x, wq, wk, wv, None, row0=3, q_pos_base=901, kv_pos_base=3)
    for g, w, H in zip(plain, (wq, wk, wv), (hq, hkv, hkv)):
        got = orc.bf16_u16_to_fp32(g).astype(np.float64).transpose(1, 0, 2).reshape(L, H * d)
        err = np.abs(got - lo.project_exact(x, w))
        bound = lo.projection_error_bound(x, w)
        assert np.all(err <= bound), float(np.max(err / bound))
    assert np.array_equal(roped[0], lo.apply_rope(plain[0], 901))
    assert np.array_equal(roped[1], lo.apply_rope(plain[1], 3)) and np.array_equal(roped[2], plain[2])
