"""The prefill chunk (config 5) on the GPU.

GEMM, Y = X W^T for T tokens on the bf16 matrix cores; two references on the
same seeded inputs:

* exact-input reference: X and the dequantized weights rounded to bf16 the
  way the kernel rounds them (Q4_K: w = d sc q - dmin m rounded once to fp32;
  Q6_K: w = (d sc) q, exact in fp32; then bf16 nearest-even), products and
  sums in fp64.  Only the kernel's fp32 accumulation order differs:
  tolerance 1e-5 relative L2.  This pins indexing, operand layouts and the
  block decodes.
* full-precision reference: fp64 GEMM of the fp32 X and the exactly
  dequantized weights (what the reference's T sequential fp32 matvecs
  approximate, engine.c:119-152).  bf16 inputs cost ~2^-9 relative per
  product: tolerance 1e-2 relative L2 (observed ~3e-3).

RoPE + append + causal attention of T tokens (the fp32-MFMA flash kernel):
the cache rows bit-exact with the oracle's RoPE, each token's attention
within 1e-5 of the oracle and of the decode kernel at its position.

Whole-model prefill (forward() over a prompt, engine.c:559-595) against T
sequential oracle steps (bit-exact with the reference's forward()): the
projections see bf16 inputs, so the last token's logits and the new cache
rows are held to 3e-2 relative L2 (observed about 5e-3) and the next greedy
token must agree."""
import ctypes as C

import numpy as np
import pytest

from guanaco_amd import spec as S
from util import bits, dequant_q4k_f64, dequant_q6k_f64, dequant_q8_0_f64, rel_l2

pytestmark = pytest.mark.gpu


def bf16_round(a):
    b = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    b = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16) << 16
    return b.astype(np.uint32).view(np.float32)


def q4k_dequant_kernel_order(w, rows, cols):
    """Per weight: fp32(d*sc*q - dmin*m) with one rounding (the kernel's
    fma), d*sc and dmin*m exact in fp32."""
    blk = w.reshape(rows, cols // 256, 144)
    d = blk[:, :, 0:2].copy().view(np.float16)[..., 0].astype(np.float64)
    dm = blk[:, :, 2:4].copy().view(np.float16)[..., 0].astype(np.float64)
    sc = blk[:, :, 4:16].astype(np.int64)
    qs = blk[:, :, 16:144].astype(np.int64)
    out = np.empty((rows, cols // 256, 256), np.float64)
    for j in range(8):
        if j < 4:
            s, m = sc[..., j] & 63, sc[..., j + 4] & 63
        else:
            s = (sc[..., j + 4] & 15) | ((sc[..., j - 4] >> 6) << 4)
            m = (sc[..., j + 4] >> 4) | ((sc[..., j] >> 6) << 4)
        chunk = qs[..., 32 * (j // 2):32 * (j // 2) + 32]
        q = (chunk >> 4) if (j & 1) else (chunk & 15)
        a = (d * s).astype(np.float32).astype(np.float64)
        mm = (dm * m).astype(np.float32).astype(np.float64)
        out[..., 32 * j:32 * j + 32] = (a[..., None] * q - mm[..., None]).astype(np.float32)
    return out.reshape(rows, cols)


SHAPES = [(64, 128, 256), (100, 256, 512), (512, 1024, 4096), (130, 384, 1024)]


@pytest.mark.parametrize("T,N,K", SHAPES)
@pytest.mark.parametrize("mode", [0, 1])
def test_prefill_gemm(ctx, orc, T, N, K, mode):
    _gemm_case(ctx, orc, S.Q4_K, T, N, K, mode)


@pytest.mark.parametrize("T,N,K", [(64, 128, 512), (100, 256, 512), (512, 1024, 4096), (77, 384, 1536),
                                   (33, 128, 3584)])
@pytest.mark.parametrize("mode", [0, 1])
def test_prefill_gemm_q6k(ctx, orc, T, N, K, mode):
    _gemm_case(ctx, orc, S.Q6_K, T, N, K, mode)


@pytest.mark.parametrize("T,N,K", [(64, 128, 256), (100, 256, 512), (512, 1024, 4096), (77, 384, 1536),
                                   (33, 128, 5632), (512, 2048, 2048)])
@pytest.mark.parametrize("mode", [0, 1])
def test_prefill_gemm_q8_0(ctx, orc, T, N, K, mode):
    """Q8_0 weights (quant_matvec_q8_0.c:5-10): w = d q is exact in fp32, so
    the exact-input reference is bf16(d q) against bf16(x)."""
    _gemm_case(ctx, orc, S.Q8_0, T, N, K, mode)


def _dequant(dtype, w, rows, cols):
    return {S.Q4_K: dequant_q4k_f64, S.Q6_K: dequant_q6k_f64, S.Q8_0: dequant_q8_0_f64}[dtype](w, rows, cols)


def _kernel_weights(dtype, w, rows, cols):
    """The fp32 weights the kernel rounds to bf16: Q4_K in its fma order,
    Q6_K and Q8_0 exact."""
    if dtype == S.Q4_K:
        return q4k_dequant_kernel_order(w, rows, cols)
    return _dequant(dtype, w, rows, cols).astype(np.float32)


def _gemm_case(ctx, orc, dtype, T, N, K, mode):
    import guanaco_amd.hip as H
    seed = (T << 20) ^ (N << 8) ^ K ^ (dtype << 28)
    w = orc.synth_quant(dtype, seed, N, K)
    x = orc.synth_normal(seed + 1, T * K).reshape(T, K)
    r = orc.synth_normal(seed + 2, T * N).reshape(T, N)
    wd, xd = ctx.upload_weight(w), ctx.upload(x)
    yd = ctx.upload(r) if mode == 1 else ctx.alloc(4 * T * N)
    rc = H.lib.gq_hip_prefill_gemm_dev(ctx.h, dtype, mode, wd, N, K, xd.ptr, T, yd.ptr,
                                       yd.ptr if mode == 1 else None)
    assert rc == 0
    y = yd.download(count=T * N).reshape(T, N)
    base = r.astype(np.float64) if mode == 1 else 0.0
    wf = _dequant(dtype, w, N, K)
    wk = _kernel_weights(dtype, w, N, K)
    exact_in = bf16_round(x).astype(np.float64) @ bf16_round(wk).astype(np.float64).T
    assert rel_l2(y, base + exact_in) < 1e-5
    full = x.astype(np.float64) @ wf.T
    e = rel_l2(y - base, full)
    assert e < 1e-2, e
    H.lib.gq_hip_free(ctx.h, wd)
    xd.free(), yd.free()


@pytest.mark.parametrize("dtype,N,K,mode", [
    (S.Q4_K, 4096, 4096, 0),    # q / o
    (S.Q4_K, 14336, 4096, 0),   # gate / up
    (S.Q4_K, 4096, 14336, 1),   # down + residual
    (S.Q6_K, 4096, 14336, 1),   # the Q6_K down of the Q4_K_M mix
    (S.Q6_K, 14336, 4096, 0),   # Q6_K gate / up: 128-token tiles from the unit layout
])
def test_prefill_gemm_config5_shapes(ctx, orc, dtype, N, K, mode):
    """Config 5's full 512-token GEMMs on the 8B projection shapes; every
    token is checked on 384 sampled output rows (first and last included)
    against the exact-input fp64 reference (1e-5) and the full-precision one
    (1e-2)."""
    import guanaco_amd.hip as H
    T = 512
    seed = 0xC0F5 ^ (N << 8) ^ K ^ (dtype << 28)
    print(f"prefill GEMM {T}x{N}x{K} dtype {dtype} mode {mode}", flush=True)
    w = orc.synth_quant(dtype, seed, N, K)
    x = orc.synth_normal(seed + 1, T * K).reshape(T, K)
    r = orc.synth_normal(seed + 2, T * N).reshape(T, N)
    wd, xd = ctx.upload_weight(w), ctx.upload(x)
    yd = ctx.upload(r) if mode == 1 else ctx.alloc(4 * T * N)
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, dtype, mode, wd, N, K, xd.ptr, T, yd.ptr,
                                         yd.ptr if mode == 1 else None) == 0
    y = yd.download(count=T * N).reshape(T, N)
    H.lib.gq_hip_free(ctx.h, wd)
    xd.free(), yd.free()
    idx = np.unique(np.concatenate([[0, N - 1], np.random.default_rng(seed).choice(N, 382, replace=False)]))
    ws = np.ascontiguousarray(w.reshape(N, -1)[idx]).reshape(-1)
    n = idx.size
    wf = dequant_q4k_f64(ws, n, K) if dtype == S.Q4_K else dequant_q6k_f64(ws, n, K)
    wk = q4k_dequant_kernel_order(ws, n, K) if dtype == S.Q4_K else wf.astype(np.float32)
    base = r[:, idx].astype(np.float64) if mode == 1 else 0.0
    ys = y[:, idx]
    exact_in = bf16_round(x).astype(np.float64) @ bf16_round(wk).astype(np.float64).T
    assert rel_l2(ys, base + exact_in) < 1e-5
    assert rel_l2(ys - base, x.astype(np.float64) @ wf.T) < 1e-2


def test_prefill_gemm_rejects_bad_shapes(ctx):
    import guanaco_amd.hip as H
    buf = ctx.alloc(1 << 20)
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, S.Q4_K, 0, buf.ptr, 100, 256, buf.ptr, 4, buf.ptr, None) != 0
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, S.Q4_K, 0, buf.ptr, 128, 300, buf.ptr, 4, buf.ptr, None) != 0
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, S.F32, 0, buf.ptr, 128, 256, buf.ptr, 4, buf.ptr, None) != 0
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, S.Q8_0, 0, buf.ptr, 128, 288, buf.ptr, 4, buf.ptr, None) != 0
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, S.Q6_K, 0, buf.ptr, 128, 256, buf.ptr, 4, buf.ptr, None) == -2
    buf.free()


def silu_mul_f32(g, u):
    g = g.astype(np.float32)
    with np.errstate(over="ignore"):
        sig = np.float32(1) / (np.float32(1) + np.exp(np.float32(0) - g))
    return (g * sig) * u.astype(np.float32)


@pytest.mark.parametrize("dtype,T,N,K", [(S.Q4_K, 512, 1024, 4096), (S.Q4_K, 70, 192, 512),
                                         (S.Q6_K, 100, 256, 1024), (S.Q6_K, 100, 256, 4096),
                                         (S.Q8_0, 100, 256, 1024), (S.Q8_0, 512, 1024, 2048)])
def test_prefill_gate_up_swiglu(ctx, orc, dtype, T, N, K):
    """gate and up in one launch with SiLU(gate) * up in the epilogue
    (kernels_cpu.c:312-389), bf16 out: against the exact-input reference
    (bf16 operands, fp64 sums, the SwiGLU in fp32 and bf16 rounding as the
    kernel does; only the accumulation order differs) and against fp64."""
    import guanaco_amd.hip as H
    seed = (T << 16) ^ (N << 4) ^ K
    wg, wu = orc.synth_quant(dtype, seed, N, K), orc.synth_quant(dtype, seed + 1, N, K)
    x = orc.synth_normal(seed + 2, T * K).reshape(T, K)
    gd, ud, xd = ctx.upload_weight(wg), ctx.upload_weight(wu), ctx.upload(x)
    act = ctx.alloc(2 * T * N)
    assert H.lib.gq_hip_prefill_gate_up_dev(ctx.h, dtype, gd, ud, N, K, xd.ptr, T, act.ptr) == 0
    a16 = act.download(np.uint16, count=T * N).reshape(T, N)
    got = (a16.astype(np.uint32) << 16).view(np.float32)
    deq = lambda w, n, k: _dequant(dtype, w, n, k)  # noqa: E731
    kern = lambda w: _kernel_weights(dtype, w, N, K)  # noqa: E731
    xb = bf16_round(x).astype(np.float64)
    g = xb @ bf16_round(kern(wg)).astype(np.float64).T
    u = xb @ bf16_round(kern(wu)).astype(np.float64).T
    assert rel_l2(got, bf16_round(silu_mul_f32(g, u))) < 1e-3
    g64, u64 = x.astype(np.float64) @ deq(wg, N, K).T, x.astype(np.float64) @ deq(wu, N, K).T
    with np.errstate(over="ignore"):
        assert rel_l2(got, g64 / (1 + np.exp(-g64)) * u64) < 2e-2
    act.free(), xd.free()
    H.lib.gq_hip_free(ctx.h, gd), H.lib.gq_hip_free(ctx.h, ud)


@pytest.mark.parametrize("T", [1, 32, 33, 64])
@pytest.mark.parametrize("dtype,N,K", [
    (S.Q4_K, 128, 256),     # one step a split, one part
    (S.Q4_K, 6144, 4096),   # the 8B q/k/v rows: 16 waves up to 32 tokens
    (S.Q4_K, 384, 14336),   # 56 steps a split over 8 or 7 parts
    (S.Q6_K, 256, 2048),    # unit layout
    (S.Q6_K, 128, 1536),    # reference layout: past 32 tokens the 64-token tiles of longer chunks
    (S.Q8_0, 640, 5632),    # 22 steps a split
])
def test_prefill_gemm_few_tokens(ctx, orc, dtype, N, K, T):
    """The shapes of up to 64 tokens (four K splits a workgroup, parts over
    the grid), stored and added to a residual, on up to 256 sampled rows
    against the exact-input fp64 product (1e-5)."""
    import guanaco_amd.hip as H
    seed = (T << 20) ^ (N << 4) ^ K ^ (dtype << 28)
    w = orc.synth_quant(dtype, seed, N, K)
    x = orc.synth_normal(seed + 1, T * K).reshape(T, K)
    r = orc.synth_normal(seed + 2, T * N).reshape(T, N)
    idx = np.unique(np.concatenate([[0, N - 1], np.random.default_rng(seed).choice(N, min(N, 254), replace=False)]))
    ws = np.ascontiguousarray(w.reshape(N, -1)[idx]).reshape(-1)
    want = bf16_round(x).astype(np.float64) @ bf16_round(_kernel_weights(dtype, ws, idx.size, K)).astype(np.float64).T
    wd, xd, yd = ctx.upload_weight(w), ctx.upload(x), ctx.upload(r)
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, dtype, 1, wd, N, K, xd.ptr, T, yd.ptr, yd.ptr) == 0
    assert rel_l2(yd.download(count=T * N).reshape(T, N)[:, idx] - r[:, idx].astype(np.float64), want) < 1e-5
    assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, dtype, 0, wd, N, K, xd.ptr, T, yd.ptr, None) == 0
    assert rel_l2(yd.download(count=T * N).reshape(T, N)[:, idx], want) < 1e-5
    xd.free(), yd.free()
    H.lib.gq_hip_free(ctx.h, wd)


@pytest.mark.parametrize("dtype,T,N,K", [(S.Q4_K, 1, 64, 256), (S.Q4_K, 32, 10240, 2048), (S.Q4_K, 64, 192, 1024),
                                         (S.Q8_0, 33, 320, 2048), (S.Q6_K, 32, 64, 512), (S.Q6_K, 64, 128, 2048)])
def test_prefill_gate_up_few_tokens(ctx, orc, dtype, T, N, K):
    """Gate/up + SwiGLU in those shapes (10240 rows: sixteen waves)."""
    test_prefill_gate_up_swiglu(ctx, orc, dtype, T, N, K)


@pytest.mark.parametrize("T,N,K", [(512, 14336, 4096), (300, 11008, 2048), (257, 11008, 1024)])
def test_prefill_gate_up_wide_tile(ctx, orc, T, N, K):
    """The fused Q4_K gate/up launch on the wide tile (64 rows per wave),
    which the launcher takes when the 128-row tiles alone fill the GPU
    (config 5's 2 x 14336 x 4096; ragged 300- and 257-token cases, the
    last with one token in its last tile).  Rows are
    independent, so each half of the rows runs again as a launch of its own,
    which on 256 CUs takes the 32-row tile without a K split (7168 rows at
    512 tokens, 5504 at 300 and 257): the same sums in the same order, so the halves
    must agree bit for bit with the wide launch.  Sampled rows are held to
    the exact-input reference as test_prefill_gate_up_swiglu does."""
    import guanaco_amd.hip as H
    seed = 0x5EED ^ (T << 16) ^ N
    print(f"prefill gate/up wide tile {T}x{N}x{K}", flush=True)
    wg, wu = orc.synth_quant(S.Q4_K, seed, N, K), orc.synth_quant(S.Q4_K, seed + 1, N, K)
    x = orc.synth_normal(seed + 2, T * K).reshape(T, K)
    gd, ud, xd = ctx.upload_weight(wg), ctx.upload_weight(wu), ctx.upload(x)
    half = N // 2
    act, sub = ctx.alloc(2 * T * N), ctx.alloc(2 * T * half)
    assert H.lib.gq_hip_prefill_gate_up_dev(ctx.h, S.Q4_K, gd, ud, N, K, xd.ptr, T, act.ptr) == 0
    wide = act.download(np.uint16, count=T * N).reshape(T, N)
    if ctx.info()[0] == 256:
        rowbytes = K // 256 * 144
        for r0 in (0, half):
            assert H.lib.gq_hip_prefill_gate_up_dev(ctx.h, S.Q4_K, gd + r0 * rowbytes, ud + r0 * rowbytes, half, K,
                                                    xd.ptr, T, sub.ptr) == 0
            narrow = sub.download(np.uint16, count=T * half).reshape(T, half)
            assert np.array_equal(wide[:, r0:r0 + half], narrow), r0
    idx = np.unique(np.concatenate([[0, N - 1], np.random.default_rng(seed).choice(N, 254, replace=False)]))
    n = idx.size
    pick = lambda w: np.ascontiguousarray(w.reshape(N, -1)[idx]).reshape(-1)  # noqa: E731
    xb = bf16_round(x).astype(np.float64)
    g = xb @ bf16_round(q4k_dequant_kernel_order(pick(wg), n, K)).astype(np.float64).T
    u = xb @ bf16_round(q4k_dequant_kernel_order(pick(wu), n, K)).astype(np.float64).T
    got = (wide[:, idx].astype(np.uint32) << 16).view(np.float32)
    assert rel_l2(got, bf16_round(silu_mul_f32(g, u))) < 1e-3
    act.free(), sub.free(), xd.free()
    H.lib.gq_hip_free(ctx.h, gd), H.lib.gq_hip_free(ctx.h, ud)


@pytest.mark.parametrize("nh,nkv,hd,pre,T,ms", [
    (32, 8, 128, 0, 512, 640),     # config 5: a 512-token chunk from position 0
    (32, 8, 128, 300, 200, 640),   # after a cached prefix
    (32, 4, 64, 5, 130, 135),      # TinyLlama shape, ends at the cache end (max_seq % 16 != 0)
    (8, 8, 64, 0, 3, 16),          # G = 1, three tokens
    (64, 8, 128, 7, 33, 64),       # G = 8, two tokens per tile
    (16, 8, 64, 1, 21, 40),        # G = 2
    # ragged tiles of the fp32 kernel
    (32, 4, 64, 77, 200, 277),     # G = 8, ragged last tile, ends at the cache end
    (32, 32, 64, 3, 190, 200),     # G = 1, 64 tokens per tile
    (32, 32, 128, 64, 129, 200),   # one token in the last tile
    (64, 8, 128, 63, 97, 160),     # the first key of a block is the last one seen
    (64, 32, 64, 0, 65, 65),       # G = 2, one token past a tile
    # the split-bf16 kernel: its keys whole
    (64, 64, 64, 0, 515, 515),     # G = 1, ragged last tile, ends at the cache end
    (64, 32, 64, 0, 1025, 1025),   # G = 2, one token past a tile
    (64, 64, 128, 0, 512, 640),    # whole tiles
    (32, 8, 128, 0, 1000, 1000),   # G = 4, ragged
    # and in parts, merged
    (32, 8, 128, 256, 512, 768),   # G = 4, two parts
    (32, 8, 128, 0, 900, 900),     # two parts, the first tile with keys in one alone
    (32, 4, 64, 2000, 257, 2257),  # G = 8, seven parts, one token past a tile
    (64, 32, 128, 1300, 130, 1430),  # G = 2, five parts
    (64, 8, 128, 1535, 33, 1600),  # eight parts, the first key of a block is the last one seen
    (32, 8, 128, 8100, 1, 8160),   # one token
])
def test_prefill_attention(ctx, orc, nh, nkv, hd, pre, T, ms):
    from oracle import HostKV, fptr
    theta = 500000.0
    ctx.kv_init(1, nkv, hd, ms, theta)
    seed_k, seed_v = 0x5EED + pre, 0xFEED + T
    if pre:
        ctx.kv_prefill_synth(seed_k, seed_v, pre)
    rng = np.random.default_rng(T * 1000 + pre)
    q = rng.standard_normal((T, nh * hd)).astype(np.float32)
    k = rng.standard_normal((T, nkv * hd)).astype(np.float32)
    v = rng.standard_normal((T, nkv * hd)).astype(np.float32)
    qb, kb, vb, ob = ctx.upload(q), ctx.upload(k), ctx.upload(v), ctx.alloc(4 * T * nh * hd)
    assert ctx.prefill_attention_dev(0, pre, T, nh, qb, kb, vb, ob) == 0
    out = ob.download(count=T * nh * hd).reshape(T, nh * hd)
    qr = qb.download(count=T * nh * hd).reshape(T, nh * hd)
    # RoPE and the appended rows bit-exact with the oracle
    kv = HostKV(1, nkv, hd, ms)
    for arr, seed in ((kv.k, seed_k), (kv.v, seed_v)):
        orc.lib.orc_synth_kv(seed, fptr(arr), 1, nkv, hd, ms, pre)
    kr = np.empty_like(k)
    for t in range(T):
        q2, k2 = orc.rope(q[t], k[t], nh, nkv, hd, pre + t, theta)
        assert np.array_equal(bits(qr[t]), bits(q2)), t
        kr[t] = k2
    kvk, kvv = kv.k.reshape(nkv, ms, hd), kv.v.reshape(nkv, ms, hd)
    kvk[:, pre:pre + T] = kr.reshape(T, nkv, hd).transpose(1, 0, 2)
    kvv[:, pre:pre + T] = v.reshape(T, nkv, hd).transpose(1, 0, 2)
    dk, dv = ctx.kv_read_layer(0)
    assert np.array_equal(bits(dk), bits(kv.k)) and np.array_equal(bits(dv), bits(kv.v))
    # each token against the oracle (fp32 throughout, only the summation
    # order differs) and against the decode kernel at its position
    q1, o1 = ctx.alloc(4 * nh * hd), ctx.alloc(4 * nh * hd)
    for t in sorted({0, 1, 2, 15, 16, 17, T // 2, T - 2, T - 1} & set(range(T))):
        ref = orc.attention(qr[t], kv, 0, nh, pre + t)
        assert rel_l2(out[t], ref) < 1e-5, t
        if nh // nkv in (1, 4, 8):  # the decode kernel's group sizes
            q1.upload(qr[t])
            assert ctx.attention_dev(0, pre + t, nh, q1, o1) == 0
            assert rel_l2(out[t], o1.download()) < 1e-5, t
    for b in (qb, kb, vb, ob, q1, o1):
        b.free()


@pytest.mark.parametrize("nh,nkv,pre,T", [(64, 64, 0, 512), (32, 8, 256, 768)])
@pytest.mark.parametrize("bad", ["none", "k_inf", "v_inf", "v_nan", "q_nan", "huge"])
def test_prefill_attention_wide_equals_narrow(ctx, bad, nh, nkv, pre, T):
    """One launch over 512 tokens (the split-bf16 kernel; after a prefix its
    keys in two parts) against the same tokens in launches of 32 (the fp32
    kernel): finite outputs to fp32 rounding, and exactly the same non-finite
    ones, for which the wide kernel has to fall back to fp32 arithmetic."""
    hd, ms = 128, T + 64
    rng = np.random.default_rng(5)
    q = rng.standard_normal((T, nh * hd)).astype(np.float32)
    k = rng.standard_normal((T, nkv * hd)).astype(np.float32)
    v = rng.standard_normal((T, nkv * hd)).astype(np.float32)
    if bad == "k_inf":
        k[70 + pre // 2, 3 * hd + 6] = np.inf
    elif bad == "v_inf":
        v[131, 2 * hd + 5] = -np.inf
    elif bad == "v_nan":
        v[9, 7 * hd + 127] = np.nan
    elif bad == "q_nan":
        q[T - 56, 11 * hd] = np.nan
    elif bad == "huge":  # rounds to an infinite bf16
        v[40, 0] = np.float32(3.4e38)
    got = []
    for wide_step in (True, False):
        ctx.kv_init(1, nkv, hd, ms, 500000.0)
        out = []
        t = 0
        while t < T:
            step = T - pre if wide_step and t >= pre else 32
            qb, kb, vb = (ctx.upload(a[t:t + step]) for a in (q, k, v))
            ob = ctx.alloc(4 * step * nh * hd)
            assert ctx.prefill_attention_dev(0, t, step, nh, qb, kb, vb, ob) == 0
            out.append(ob.download(count=step * nh * hd).reshape(step, nh * hd))
            for b in (qb, kb, vb, ob):
                b.free()
            t += step
        got.append(np.concatenate(out))
    wide, narrow = got
    assert np.array_equal(np.isnan(wide), np.isnan(narrow))
    fin = np.isfinite(narrow)
    assert np.array_equal(np.isfinite(wide), fin) and np.array_equal(wide[~fin & ~np.isnan(wide)], narrow[~fin & ~np.isnan(wide)])
    assert np.isnan(narrow).any() == (bad not in ("none", "huge"))
    if bad != "huge":
        assert rel_l2(wide[fin], narrow[fin]) < 2e-6
    else:  # the column that holds it, and the rest
        c = np.abs(narrow).max(axis=0) > 1e30
        assert c.any() and rel_l2(wide[:, c] / 1e30, narrow[:, c] / 1e30) < 2e-6 and rel_l2(wide[:, ~c], narrow[:, ~c]) < 2e-6


def test_prefill_attention_rejects_bad_positions(ctx):
    ctx.kv_init(1, 2, 64, 32, 500000.0)
    b = ctx.alloc(4 * 40 * 8 * 64)
    assert ctx.prefill_attention_dev(0, 30, 3, 8, b, b, b, b) == -5
    assert ctx.prefill_attention_dev(0, -1, 3, 8, b, b, b, b) == -5
    assert ctx.prefill_attention_dev(0, 0, 0, 8, b, b, b, b) == -1
    assert ctx.prefill_attention_dev(0, 0, 3, 7, b, b, b, b) == -1
    b.free()


@pytest.mark.parametrize("nh,nkv,hd", [(32, 1, 64), (6, 2, 64), (32, 2, 128), (8, 4, 96)])
def test_prefill_attention_rejects_unsupported_heads(ctx, nh, nkv, hd):
    """Head geometries that no kernel takes (more than 8 query heads per KV
    head, 3, or head_dim 96) are refused, and the cache is left as it was."""
    ctx.kv_init(1, nkv, hd, 64, 500000.0)
    ctx.kv_prefill_synth(5, 6, 64)
    before = ctx.kv_read_layer(0)
    b = ctx.alloc(4 * 40 * nh * hd)
    for T, pos in ((1, 0), (37, 20)):
        assert ctx.prefill_attention_dev(0, pos, T, nh, b, b, b, b) == -1
    for d, e in zip(ctx.kv_read_layer(0), before):
        assert np.array_equal(bits(d), bits(e))
    b.free()


PF_TOL = 3e-2


@pytest.mark.parametrize("pre,T,ms", [(0, 48, 64), (24, 39, 64), (0, 600, 640)])
def test_prefill_model_vs_oracle(ctx, orc, pre, T, ms):
    """forward() over a T-token prompt at pos `pre` (the reference's own
    prefill call, generate.c:200-226), then one decode step from it."""
    import guanaco_amd.hip as H
    from oracle import HostModel
    from guanaco_amd.synth import tensor_seed
    spec = S.TINY_TEST
    hm = HostModel(orc, spec, ms)
    dm = H.DeviceModel(ctx, spec, ms, prefill=pre)
    kv = hm.new_kv()
    if pre:
        kv.prefill(orc, spec, pre)
    rng = np.random.default_rng(T + pre)
    toks = rng.integers(0, spec.vocab, T).astype(np.int32)
    nxt, lg, hid, ms_dev = dm.prefill(toks, pre, want_hidden=True)
    for t in range(T):
        t_cpu, lc, _ = hm.forward(kv, int(toks[t]), pre + t)
    assert rel_l2(lg, lc) < PF_TOL
    assert nxt == t_cpu
    for l in range(spec.n_layers):
        dk, dv = ctx.kv_read_layer(l)
        for d, h in ((dk, kv.view("k")[l]), (dv, kv.view("v")[l])):
            d = d.reshape(h.shape)
            assert np.array_equal(d[:, :pre], h[:, :pre])          # the cached prefix untouched
            assert rel_l2(d[:, pre:pre + T], h[:, pre:pre + T]) < PF_TOL
    # decode continues from the prefilled cache
    t_gpu, lg2, _ = dm.forward(nxt, pre + T)
    t_cpu2, lc2, _ = hm.forward(kv, t_cpu, pre + T)
    assert rel_l2(lg2, lc2) < PF_TOL and t_gpu == t_cpu2
    print(f"prefill T={T} pre={pre}: logits rel {rel_l2(lg, lc):.2e}, device {ms_dev:.3f} ms")


@pytest.mark.parametrize("T,N,K,mode", [(96, 256, 4096, 0), (77, 384, 2048, 1), (512, 4096, 14336, 1)])
def test_prefill_q6k_unit_layout_vs_reference_layout(ctx, orc, T, N, K, mode):
    """Q6_K weights whose rows fall on 16-byte boundaries (K % 2048 == 0) go
    through the GEMM in the decode matvec's unit layout (a copy made per call
    here; a bound model reads the copy model bind made for the decode step):
    the same bf16 weights as the reference layout, which matvec path 3
    reads, summed in another K order.  The two agree to the accumulation
    order (1e-5, as against the exact-input reference) and are not the same
    bits, so the unit layout was read."""
    import guanaco_amd.hip as H
    seed = 0x5E9 ^ (T << 16) ^ (N << 4) ^ K
    w = orc.synth_quant(S.Q6_K, seed, N, K)
    x = orc.synth_normal(seed + 1, T * K).reshape(T, K)
    r = orc.synth_normal(seed + 2, T * N).reshape(T, N)
    wd, xd = ctx.upload_weight(w), ctx.upload(x)
    out = {}
    for path in ("auto", "auto_q6k_ref"):
        yd = ctx.upload(r) if mode == 1 else ctx.alloc(4 * T * N)
        with H.matvec_path(path):
            assert H.lib.gq_hip_prefill_gemm_dev(ctx.h, S.Q6_K, mode, wd, N, K, xd.ptr, T, yd.ptr,
                                                 yd.ptr if mode == 1 else None) == 0
        out[path] = yd.download(count=T * N)
        yd.free()
    assert np.abs(out["auto"]).sum() > 0
    assert rel_l2(out["auto"], out["auto_q6k_ref"]) < 1e-5
    assert not np.array_equal(bits(out["auto"]), bits(out["auto_q6k_ref"]))
    H.lib.gq_hip_free(ctx.h, wd)
    xd.free()


def test_prefill_q6k_unit_layout_model(orc):
    """A model whose Q6_K projections (v, o, down) have K % 2048 == 0 prefills
    from the unit-layout copies made at model bind (the down projection's is
    the decode step's own): logits and the last hidden state within 2e-3 of
    the reference layout's (matvec path 3; the K order of the sums differs,
    and the bf16 activations may round apart), and the prompt against the
    oracle as for the other models, on both."""
    import guanaco_amd.hip as H
    from oracle import HostModel
    spec = S.ModelSpec("q6k-steps-test", n_layers=2, hidden=2048, ff=4096, n_heads=16, n_kv_heads=4, vocab=1000,
                       layer_dtypes=dict(wv=S.Q6_K, wo=S.Q6_K, wd=S.Q6_K))
    c = H.Context(0)
    try:
        hm = HostModel(orc, spec, 64)
        dm = H.DeviceModel(c, spec, 64)
        toks = np.random.default_rng(7).integers(0, spec.vocab, 40).astype(np.int32)
        res = {}
        for path in ("auto", "auto_q6k_ref"):
            with H.matvec_path(path):
                res[path] = dm.prefill(toks, 0, want_hidden=True)
        (nxt, lg, hg, _), (nxt2, lg2, hg2, _) = res["auto"], res["auto_q6k_ref"]
        assert rel_l2(lg, lg2) < 2e-3 and rel_l2(hg, hg2) < 2e-3
        kv = hm.new_kv()
        for t in range(len(toks)):
            t_cpu, lc, _ = hm.forward(kv, int(toks[t]), t)
        assert rel_l2(lg, lc) < PF_TOL and rel_l2(lg2, lc) < PF_TOL and nxt == t_cpu and nxt2 == t_cpu
        print(f"unit layout vs reference layout: logits {rel_l2(lg, lg2):.2e}, hidden {rel_l2(hg, hg2):.2e}")
    finally:
        c.close()


def test_prefill_q8_0_model(orc):
    """A model with every weight Q8_0 prefills through the GEMM (the
    reference's prefill takes Q8_0 through linear_dispatch,
    engine.c:119-152): last-token logits and the new cache rows against T
    sequential oracle steps (PF_TOL), the next greedy token equal, and the
    result not the token-by-token one (prefill mode 1), which is held to
    the decode tolerance."""
    import guanaco_amd.hip as H
    from oracle import HostModel
    spec = S.ModelSpec("tiny-q8_0", n_layers=2, hidden=512, ff=1024, n_heads=8, n_kv_heads=2, vocab=1000,
                       layer_dtypes={k: S.Q8_0 for k in S.LAYER_WEIGHTS}, embed_dtype=S.Q8_0,
                       lm_head_dtype=S.Q8_0)
    c = H.Context(0)
    try:
        hm = HostModel(orc, spec, 64)
        dm = H.DeviceModel(c, spec, 64)
        toks = np.random.default_rng(8).integers(0, spec.vocab, 48).astype(np.int32)
        kv = hm.new_kv()
        for t in range(len(toks)):
            t_cpu, lc, _ = hm.forward(kv, int(toks[t]), t)
        nxt, lg, _, _ = dm.prefill(toks, 0)
        assert rel_l2(lg, lc) < PF_TOL and nxt == t_cpu
        for l in range(spec.n_layers):
            dk, dv = c.kv_read_layer(l)
            for d, h in ((dk, kv.view("k")[l]), (dv, kv.view("v")[l])):
                d = d.reshape(h.shape)
                assert rel_l2(d[:, :len(toks)], h[:, :len(toks)]) < PF_TOL
        assert H.lib.gq_hip_set_prefill_mode(c.h, 1) == 0
        nxt1, lg1, _, _ = dm.prefill(toks, 0)
        assert rel_l2(lg1, lc) < 1e-3 and nxt1 == t_cpu
        assert not np.array_equal(bits(lg), bits(lg1))  # the GEMM path ran in mode 0
        print(f"Q8_0 model prefill: GEMM {rel_l2(lg, lc):.2e}, token by token {rel_l2(lg1, lc):.2e}")
    finally:
        c.close()


def test_prefill_after_rebinding_larger_models(orc):
    """One context binds a small model and prefills, then binds models with
    a wider FFN and a wider hidden size and prefills again: the prefill
    workspace is sized for the model bound last (it had kept the first
    model's sizes), each prompt against the oracle."""
    import guanaco_amd.hip as H
    from oracle import HostModel
    wide_h = S.ModelSpec("tiny-wide-hidden", n_layers=2, hidden=1024, ff=2048, n_heads=16, n_kv_heads=4,
                         vocab=1000, layer_dtypes=S._q6k_on_even)
    c = H.Context(0)
    try:
        for spec in (S.TINY_TEST, S.WIDE_FF_TEST, wide_h, S.TINY_TEST):
            print(f"prefill on a rebound context: {spec.name}", flush=True)
            hm = HostModel(orc, spec, 64)
            dm = H.DeviceModel(c, spec, 64)
            toks = np.random.default_rng(spec.hidden + spec.ff).integers(0, spec.vocab, 40).astype(np.int32)
            nxt, lg, _, _ = dm.prefill(toks, 0)
            kv = hm.new_kv()
            for t in range(len(toks)):
                t_cpu, lc, _ = hm.forward(kv, int(toks[t]), t)
            assert rel_l2(lg, lc) < PF_TOL and nxt == t_cpu, spec.name
    finally:
        c.close()


def test_prefill_token_by_token_fallback(ctx, orc):
    """A model whose Q6_K projections have cols % 512 != 0 (hidden 768) is
    not taken by the GEMM: the prefill runs the decode step per token, so
    it matches the decode path (and the oracle) to the decode tolerance."""
    import guanaco_amd.hip as H
    from oracle import HostModel
    spec = S.ModelSpec("tiny-fallback", n_layers=2, hidden=768, ff=1536, n_heads=12, n_kv_heads=3, vocab=1000,
                       layer_dtypes=S._q6k_on_even)
    hm = HostModel(orc, spec, 64)
    dm = H.DeviceModel(ctx, spec, 64)
    toks = np.random.default_rng(3).integers(0, spec.vocab, 20).astype(np.int32)
    nxt, lg, _, _ = dm.prefill(toks, 0)
    kv = hm.new_kv()
    for t in range(len(toks)):
        t_cpu, lc, _ = hm.forward(kv, int(toks[t]), t)
    assert rel_l2(lg, lc) < 1e-3 and nxt == t_cpu


def test_prefill_model_rejects_bad_input(ctx):
    import guanaco_amd.hip as H
    dm = H.DeviceModel(ctx, S.TINY_TEST, 64)
    with pytest.raises(H.HipError):
        dm.prefill(np.arange(10, dtype=np.int32), 60)      # past the cache
    with pytest.raises(H.HipError):
        dm.prefill(np.array([1, 2, 5000], np.int32), 0)    # token out of range


@pytest.mark.parametrize("T", [256, 257, 511, 700])
@pytest.mark.parametrize("mix", ["q4_k_m", "q8_0"])
def test_prefill_dense_copy_vs_quantized(orc, T, mix):
    """Chunks of more than 256 tokens multiply by bf16 copies of the weights,
    made by the first such prompt; matvec path 3 dequantizes the same weights
    as it multiplies, as both do for 256 tokens.  Layer 0's V rows are that
    GEMM's own output: the same products in another order (1e-5).  After it the
    bf16 activations may round apart: 2e-3, as between the layouts above.
    128-row K and V segments (half a tile), a gate/up of 10 tiles, ragged token
    tiles."""
    import guanaco_amd.hip as H
    dts = {k: S.Q8_0 for k in S.LAYER_WEIGHTS} if mix == "q8_0" else dict(wv=S.Q6_K, wd=S.Q6_K)
    spec = S.ModelSpec("dense-test", n_layers=2, hidden=512, ff=1280 if mix == "q8_0" else 1536, n_heads=8, n_kv_heads=2,
                       vocab=1000, layer_dtypes=dts, q4k_zero_mean=True, norm_shift=4)
    c = H.Context(0)
    try:
        dm = H.DeviceModel(c, spec, 768)
        toks = np.random.default_rng(T).integers(0, spec.vocab, T).astype(np.int32)
        res = {}
        for path in ("auto_q6k_ref", "auto"):
            with H.matvec_path(path):
                _, lg, hid, _ = dm.prefill(toks, 0, want_hidden=True)
            assert (H.lib.gq_hip_prefill_copy_bytes(c.h) > 0) == (path == "auto" and T > 256)
            k0, v0 = c.kv_read_layer(0)
            res[path] = lg, hid, v0
        a, b = res["auto"], res["auto_q6k_ref"]
        v = [r[2].reshape(2, 768, 64)[:, :T] for r in (a, b)]
        assert rel_l2(v[0], v[1]) < 1e-5  # the same bits where both take as many K parts
        assert rel_l2(a[0], b[0]) < 2e-3 and rel_l2(a[1], b[1]) < 2e-3
        print(f"dense copy vs quantized, T={T}: V rows {rel_l2(v[0], v[1]):.2e}, logits {rel_l2(a[0], b[0]):.2e}")
    finally:
        c.close()


def test_prefill_dense_copy_after_a_failed_allocation(orc):
    """An allocation that the card could not hold even without the bf16 copies
    leaves them, and the bits of later prompts, as they were."""
    import guanaco_amd.hip as H
    spec = S.ModelSpec("dense-back", n_layers=2, hidden=512, ff=1536, n_heads=8, n_kv_heads=2, vocab=1000,
                       layer_dtypes=dict(wv=S.Q6_K, wd=S.Q6_K), q4k_zero_mean=True, norm_shift=4)
    c = H.Context(0)
    try:
        dm = H.DeviceModel(c, spec, 512)
        toks = np.random.default_rng(3).integers(0, spec.vocab, 300).astype(np.int32)
        with H.matvec_path("auto_q6k_ref"):
            ref = dm.prefill(toks, 0)[1]
        assert H.lib.gq_hip_prefill_copy_bytes(c.h) == 0
        with_copy = dm.prefill(toks, 0)[1]
        held = H.lib.gq_hip_prefill_copy_bytes(c.h)
        with pytest.raises(H.HipError):
            c.alloc(1 << 46)
        assert H.lib.gq_hip_prefill_copy_bytes(c.h) == held > 0
        after = dm.prefill(toks, 0)[1]
        assert np.array_equal(bits(after), bits(with_copy)) and rel_l2(with_copy, ref) < 2e-3
    finally:
        c.close()


def test_prefill_weights_rewritten_in_place(orc):
    """A Q8_0 model whose weights are written again in place after it was
    bound: a prompt of 300 tokens sees the new ones, as a model bound after the
    write does (2e-3, as between the kernels above), and not the copy of the
    old ones."""
    import guanaco_amd.hip as H
    spec = S.ModelSpec("dense-rewrite", n_layers=2, hidden=512, ff=1024, n_heads=8, n_kv_heads=2, vocab=1000,
                       layer_dtypes={k: S.Q8_0 for k in S.LAYER_WEIGHTS}, embed_dtype=S.Q8_0, lm_head_dtype=S.Q8_0)
    toks = np.random.default_rng(4).integers(0, spec.vocab, 300).astype(np.int32)
    c = H.Context(0)
    try:
        dm = H.DeviceModel(c, spec, 512)
        old = dm.prefill(toks, 0)[1]
        for l, k in ((0, "wv"), (1, "wd")):
            w = dm.weight(l, k)
            new = orc.synth_quant(S.Q8_0, 99 + l, w.rows, w.cols)
            c.check(H.lib.gq_hip_h2d(c.h, w.data, new.ctypes.data, new.nbytes), "h2d")
        got = dm.prefill(toks, 0)[1]
        c.check(H.lib.gq_hip_model_bind(c.h, C.byref(dm.model)), "model_bind")
        ref = dm.prefill(toks, 0)[1]
        assert rel_l2(got, ref) < 2e-3 and rel_l2(old, ref) > 0.1
    finally:
        c.close()


class DnArgs(C.Structure):  # gq_internal.h
    _fields_ = [("x", C.c_void_p), ("w", C.c_void_p), ("act", C.c_void_p), ("y", C.c_void_p * 3), ("rows", C.c_int * 3),
                ("nseg", C.c_int), ("T", C.c_int), ("K", C.c_int), ("part", C.c_void_p), ("part_cap", C.c_size_t),
                ("kparts", C.c_int), ("rows_total", C.c_int), ("to_parts", C.c_bool), ("kparts_out", C.c_void_p)]


class DnShape(C.Structure):
    _fields_ = [("tm", C.c_int), ("kparts", C.c_int)]


def dense_lib():
    """The launchers of gq_dense.hip, which no entry point reaches alone."""
    import guanaco_amd.hip as H
    lib = C.CDLL(H.LIB_PATH)
    shape, tile, size, run = (lib._Z14gq_dense_shapeiimiimi, lib._Z20gq_launch_dense_tilePviPKvS1_iiP12ihipStream_t,
                              lib._Z14gq_dense_bytesiib, lib._Z15gq_launch_denseiRK6DnArgsiP12ihipStream_t)
    shape.restype, shape.argtypes = DnShape, [C.c_int, C.c_int, C.c_size_t, C.c_int, C.c_int, C.c_size_t, C.c_int]
    tile.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p]
    size.restype, size.argtypes = C.c_size_t, [C.c_int, C.c_int, C.c_bool]
    run.argtypes = [C.c_int, C.POINTER(DnArgs), C.c_int, C.c_void_p]
    return shape, tile, size, run, lib.hipDeviceSynchronize


STORE, RESID, SWIGLU = 0, 1, 2


@pytest.mark.parametrize("mode,dtype,rows,T,K,tm,kparts", [
    (STORE, S.Q8_0, (2048, 256, 256), 513, 512, 2, 1), (STORE, S.Q4_K, (2048, 256, 256), 257, 512, 2, 2),
    (STORE, S.Q6_K, (384,), 300, 512, 2, 4),           (STORE, S.Q4_K, (4096, 1024, 1024), 1500, 512, 4, 1),
    (STORE, S.Q6_K, (4096, 1024, 1024), 700, 4096, 4, 2), (STORE, S.Q8_0, (4096, 1024, 1024), 257, 4096, 4, 4),
    (RESID, S.Q4_K, (2048,), 700, 512, 2, 1),          (RESID, S.Q8_0, (2048,), 513, 512, 2, 2),
    (RESID, S.Q6_K, (384,), 257, 1024, 2, 4),          (RESID, S.Q4_K, (6144,), 1500, 512, 4, 1),
    (RESID, S.Q6_K, (8192,), 513, 4096, 4, 2),         (RESID, S.Q4_K, (6144,), 300, 4096, 4, 4),
    (SWIGLU, S.Q8_0, (1280,), 257, 512, 2, 1),         (SWIGLU, S.Q4_K, (14336,), 257, 512, 4, 1),
    (SWIGLU, S.Q6_K, (7168,), 513, 512, 4, 1),
])
def test_dense_gemm_shapes(ctx, orc, mode, dtype, rows, T, K, tm, kparts):
    """The GEMM on bf16 copies at each tile height, number of K parts and
    output that its rule picks (256 CUs), ragged tokens and half tiles among
    them: against fp64 sums of the same bf16 operands.  fp32 accumulation over
    K products differs by at most K 2^-24 of the sum of their magnitudes, and as
    a random walk by far less: 1e-5 of the output's 2-norm, and no element off by
    more than 1e-4 of the rms.  Nothing past the last token is written."""
    import guanaco_amd.hip as H
    shape, tile, size, run, wait = dense_lib()
    if ctx.info()[0] != 256:
        pytest.skip("the shapes are picked for 256 CUs")
    per = 128 if mode == SWIGLU else 256
    n, tiles = sum(rows), sum((r + per - 1) // per for r in rows)
    cap = 4 * T * n
    f = shape(mode, tiles, n, T, K, cap, 256)
    assert (f.tm, f.kparts) == (tm, kparts)
    print(f"dense GEMM mode {mode} rows {rows} T {T} K {K}: tm {tm}, {kparts} parts", flush=True)
    seed = 0xDE ^ (T << 16) ^ (n << 4) ^ K
    x = bf16_round(orc.synth_normal(seed, T * K).reshape(T, K))
    ws = [orc.synth_quant(dtype, seed + 1 + i, r, K) for i, r in enumerate(rows * (2 if mode == SWIGLU else 1))]
    exact = [x.astype(np.float64) @ bf16_round(_kernel_weights(dtype, w, w_rows, K)).astype(np.float64).T
             for w, w_rows in zip(ws, rows * (2 if mode == SWIGLU else 1))]
    bufs = [ctx.upload((x.view(np.uint32) >> 16).astype(np.uint16))]
    wd = [ctx.upload_weight(w) for w in ws]
    copy = ctx.alloc(sum(size(r, K, mode == SWIGLU) for r in rows))
    part = ctx.alloc(4 * cap)
    at = 0
    for i, r in enumerate(rows):
        assert tile(copy.ptr + at, dtype, wd[i], wd[1] if mode == SWIGLU else None, r, K, None) == 0
        at += size(r, K, mode == SWIGLU)
    a = DnArgs(x=bufs[0].ptr, w=copy.ptr, nseg=len(rows), T=T, K=K, part=part.ptr, part_cap=cap)
    a.rows[:len(rows)] = rows
    if mode == SWIGLU:
        act = ctx.upload(np.full((T + 8, n), 0x7e57, np.uint16))
        a.act = act.ptr
        assert run(mode, C.byref(a), 256, None) == 0 and wait() == 0
        got16 = act.download(np.uint16).reshape(T + 8, n)
        got = (got16[:T].astype(np.uint32) << 16).view(np.float32)
        assert (got16[T:] == 0x7e57).all()
        ref = bf16_round(silu_mul_f32(exact[0], exact[1]))
        assert rel_l2(got, ref) < 1e-3  # a sum that rounds the other way is off by one in 2^8
        assert np.abs(got - ref).max() <= 2.0 ** -7 * np.abs(ref).max()
        bufs += [act]
    else:
        old = [orc.synth_normal(seed + 9 + i, (T + 8) * r).reshape(T + 8, r) for i, r in enumerate(rows)]
        ys = []
        for leave in (False, True):  # whether the caller adds the parts
            yd = [ctx.upload(o) for o in old]
            for i, b in enumerate(yd):
                a.y[i] = b.ptr
            left = C.c_int(-1)
            a.kparts_out = C.addressof(left) if leave else None
            assert run(mode, C.byref(a), 256, None) == 0 and wait() == 0
            y = [b.download().reshape(T + 8, r) for b, r in zip(yd, rows)]
            for b, o in zip(y, old):
                assert np.array_equal(bits(b[T:]), bits(o[T:]))
            to_parts = mode == RESID or kparts > 1
            if leave:
                assert left.value == (kparts if to_parts else 0)
            if leave and to_parts:
                s = part.download(count=kparts * T * n).reshape(kparts, T, n).astype(np.float64).sum(0)
                for b, o in zip(y, old):
                    assert np.array_equal(bits(b), bits(o))  # y is left to the caller
                y = [s[:, sum(rows[:i]):sum(rows[:i + 1])] + (old[i][:T] if mode == RESID else 0) for i in range(len(rows))]
            ys.append([b[:T] for b in y])
            for b in yd:
                b.free()
        for y in ys:
            for got, ref, o in zip(y, exact, old):
                ref = ref + o[:T] if mode == RESID else ref
                assert rel_l2(got, ref) < 1e-5
                assert np.abs(got - ref).max() < 1e-4 * np.sqrt(np.mean(ref ** 2))
    for b in bufs + [copy, part]:
        b.free()
    for w in wd:
        H.lib.gq_hip_free(ctx.h, w)


@pytest.mark.parametrize("T,step", [(37, 37), (300, 300), (2049, 1025), (4097, 1366), (8200, 1640)])
def test_prompt_over_chunks_equals_calls(T, step):
    """A prompt longer than a chunk (2048 tokens) runs in equal chunks, the
    last one ragged, whose tokens wait in pinned memory for 8192: the same
    bits, cache rows included, as those chunks given one call each, and again
    when it is repeated (as is a shorter one)."""
    import guanaco_amd.hip as H
    spec = S.ModelSpec("chunks", n_layers=2, hidden=512, ff=1024, n_heads=8, n_kv_heads=2, vocab=1000,
                       layer_dtypes=dict(wv=S.Q6_K, wd=S.Q6_K), q4k_zero_mean=True, norm_shift=4)
    c = H.Context(0)
    try:
        dm = H.DeviceModel(c, spec, 8448)
        toks = np.random.default_rng(T).integers(0, spec.vocab, T).astype(np.int32)
        got = []
        for n in (step, T, T):
            for t in range(0, T, n):
                nxt, lg, hid, _ = dm.prefill(toks[t:t + n], t, want_hidden=True)
            kv = [r.reshape(2, 8448, 64)[:, :T] for l in range(2) for r in c.kv_read_layer(l)]
            got.append([np.array([nxt], np.float32), lg, hid, *kv])
        assert (H.lib.gq_hip_prefill_copy_bytes(c.h) > 0) == (T > 256)
        for other in got[1:]:
            for a, b in zip(other, got[0]):
                assert np.array_equal(bits(a), bits(b))
    finally:
        c.close()
