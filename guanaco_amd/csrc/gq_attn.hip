/*
 * gq_attn.hip — fused RoPE + KV append and split-K single-query GQA
 * attention over the device KV cache (gfx950).
 *
 * KV layout is the reference's: [layer][kv_head][max_seq][head_dim] fp32, K
 * and V in separate slabs (kv_cache.c:25-32, :90-93).
 *
 * rope_append: one workgroup rotates every Q head and the new K row with the
 * (cos, sin) table row of `pos` (precomputed on the host with the reference's
 * fp32 expressions, kernels_cpu.c:409-413; rotation products and differences
 * rounded separately, :415-429) and writes K and V at row pos of the slab
 * (kv_cache.c:101-125 with pos < max_seq; the device cache does not wrap,
 * the host rejects pos >= max_seq with -5 and the kernel returns for such a
 * position).  Appended rows are bit copies of the reference's.
 *
 * attention: flash-decoding split over the sequence.  Workgroup (g, c)
 * streams chunk c of KV head g once for all G = n_heads/n_kv query heads
 * that share it (the reference re-reads K/V per Q head, engine.c:458-509):
 *   phase 1  scores s[h][j] = (q_h . K_j) * 1/sqrt(hd); 16 lanes per
 *            position (hd 128), 8 dims per lane, DPP row reduction;
 *   phase 2  per head chunk max m, p = expf(s - m), l = sum p;
 *   phase 3  o[h][:] = sum_j p[h][j] V_j, V read as coalesced 512-byte rows.
 * A merge kernel combines the chunks: M = max m_c, out = sum o_c e^(m_c-M) /
 * sum l_c e^(m_c-M).  The position count is read on the device, so the same
 * launch serves every step of a captured decode graph.
 *
 * Causal attention of a prompt's chunk (many query tokens): flash_prefill on
 * the fp32 matrix cores, flash_split on the bf16 ones from exact three-way
 * splits of the fp32 operands, whichever flash_shape finds the faster; see the
 * kernels.
 */
#include <algorithm>
#include <cmath>

#include "gq_device.h"
#include "gq_internal.h"

namespace {

constexpr int kThreads = 256;

__global__ __launch_bounds__(kThreads) void rope_append_kernel(RopeArgs a) {
#pragma clang fp contract(off)
  /* token blockIdx.x / n_kv of a chunk (0 for one token), KV head
   * g = blockIdx.x % n_kv and its G query heads: workgroup L runs on XCD
   * L mod 8, so head g's K/V rows are written where the flash kernel, which
   * takes head g on those workgroups, reads them */
  const int tz = (int)blockIdx.x / a.n_kv, g = (int)blockIdx.x % a.n_kv, G = a.n_heads / a.n_kv;
  const int pos = (a.pos_dev ? *a.pos_dev : a.pos) + tz;
  /* the host rejects positions outside the cache; this keeps a stray
   * device-side position from indexing past the table or the slab */
  if (pos < 0 || pos >= a.max_seq) return;
  const int half = a.hd >> 1;
  const int p = pos;
  const float2 *cs = a.cs + (size_t)pos * half;
  float *q = a.q + (size_t)tz * a.q_stride;
  const float *kin = a.k + (size_t)tz * a.k_stride, *vin = a.v + (size_t)tz * a.v_stride;
  /* element o of this token's q | k | v from the GEMM's parts, summed in
   * pg_parts_kernel's order */
  const int qd = a.n_heads * a.hd, kvd = a.n_kv * a.hd;
  const float *prow = a.parts ? a.parts + (size_t)tz * a.prow : nullptr;
  /* element pairs (2i, 2i + 1) move as one 8-byte access when every address
   * of this token allows it (always, from the runtime's own buffers: hd and
   * the strides are even); op-level callers' 4-byte-aligned buffers take
   * two scalar accesses.  The values and their order are the same. */
  const bool v2 = ((uintptr_t)q & 7) == 0 && (((uintptr_t)a.kc | (uintptr_t)a.vc) & 7) == 0 &&
                  (prow ? ((uintptr_t)prow & 7) == 0 && (a.pstride & 1) == 0
                        : (((uintptr_t)kin | (uintptr_t)vin) & 7) == 0);
  auto ld2 = [&](const float *s) {
    return v2 ? gld<float2>(s) : make_float2(s[0], s[1]);
  };
  auto st2 = [&](float *d, float2 y) {
    if (v2) gst<float2>(d, y);
    else d[0] = y.x, d[1] = y.y;
  };
  auto part2 = [&](int o) {
    float2 v = ld2(prow + o);
    for (int k = 1; k < a.kparts; k++) {
      const float2 u = ld2(prow + (size_t)k * a.pstride + o);
      v.x += u.x, v.y += u.y;
    }
    return v;
  };
  for (int t = threadIdx.x; t < (G + 1) * half; t += kThreads) {
    const bool isq = t < G * half;
    const int u = isq ? t : t - G * half;
    const int hl = u / half, i = u - hl * half;
    const int h = isq ? g * G + hl : g;
    const float2 c = cs[i];
    const float2 x = prow ? part2((isq ? 0 : qd) + h * a.hd + 2 * i)
                          : ld2((isq ? (const float *)q : kin) + (size_t)h * a.hd + 2 * i);
    const float2 y = make_float2(x.x * c.x - x.y * c.y, x.x * c.y + x.y * c.x);
    st2(isq ? q + (size_t)h * a.hd + 2 * i : a.kc + ((size_t)h * a.max_seq + p) * a.hd + 2 * i, y);
  }
  for (int d = 2 * threadIdx.x; d < a.hd; d += 2 * kThreads) {
    const int t = g * a.hd + d;
    st2(a.vc + ((size_t)g * a.max_seq + p) * a.hd + d, prow ? part2(qd + kvd + t) : ld2(vin + t));
  }
}

/* Positions per split-K chunk (one workgroup), chosen by the cache
 * capacity.  32 gives 2080 workgroups at the 8B shape and ctx 8192 (79
 * VGPRs, six waves per SIMD): measured in the graph-replayed decode step
 * 0.9% faster than 64 (four workgroups per CU), although the attention op
 * alone, launched back to back, is 0.4 us slower; 64 had in turn measured
 * 1.3% faster per step than 128.  Past 12288 positions the merge, which
 * reads every chunk's partials, grows enough that 128 wins (16384: 32.7 vs
 * 34.7 us per layer with 64; 32768: 57.0 vs 61.9). */
int chunk_for(int max_seq) { return max_seq > 12288 ? 128 : 32; }

/* Workgroup (g, c) handles positions [Sc, Sc + S) of KV head g for the G
 * query heads sharing it.  Every K and V load of the chunk is issued before
 * any arithmetic (S/2 + S/2 VGPRs per thread at head_dim 128), so a
 * workgroup costs one memory round trip plus its FMAs. */
template <int HD, int G, int S>
__device__ __forceinline__ void attn_partial_body(const AttnArgs &a) {
  constexpr int LPP = HD / 8;          /* lanes per position, phase 1 */
  constexpr int PPI = kThreads / LPP;  /* positions per pass, phase 1 */
  constexpr int KIT = S / PPI;
  constexpr int DG = HD / 4;           /* float4 columns of a V row */
  constexpr int NPG = kThreads / DG;   /* position groups, phase 3 */
  constexpr int VIT = S / NPG;
  __shared__ float ss[G][S];
  __shared__ float4 sr[NPG][G][DG];

  const int g = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int pos = a.pos_dev ? gld<int>(a.pos_dev) : a.pos;
  const int L = min(pos + 1, a.max_seq);
  const int c0 = c * S;
  const int n = min(S, L - c0);
  if (n <= 0) return; /* past the sequence: the merge reads chunks < ceil(L/S) */
  const int h0 = g * G;
  const float *K = a.k + ((size_t)g * a.max_seq + c0) * HD;
  const float *V = a.v + ((size_t)g * a.max_seq + c0) * HD;

  /* V rows of phase 3 first: they do not depend on the scores */
  const int dg = tid % DG, pg = tid / DG;
  float4 vr[VIT];
#pragma unroll
  for (int k = 0; k < VIT; k++) vr[k] = gld_nt<float4>(V + (size_t)min(pg + NPG * k, n - 1) * HD + 4 * dg);
  /* query slices and K rows of phase 1 */
  const int sub = tid % LPP, pw = tid / LPP;
  const int d0 = 4 * sub, d1 = HD / 2 + 4 * sub;
  float4 qa[G], qb[G];
#pragma unroll
  for (int h = 0; h < G; h++) {
    qa[h] = gld<float4>(a.q + (size_t)(h0 + h) * HD + d0);
    qb[h] = gld<float4>(a.q + (size_t)(h0 + h) * HD + d1);
  }
  float4 ka[KIT], kb[KIT];
#pragma unroll
  for (int k = 0; k < KIT; k++) {
    const float *kr = K + (size_t)min(pw + PPI * k, n - 1) * HD;
    ka[k] = gld_nt<float4>(kr + d0);
    kb[k] = gld_nt<float4>(kr + d1);
  }

  /* phase 1: scores (q . k) * 1/sqrt(hd) */
#pragma unroll
  for (int k = 0; k < KIT; k++) {
    const int j = pw + PPI * k;
#pragma unroll
    for (int h = 0; h < G; h++) {
      float s = qa[h].x * ka[k].x;
      s = __builtin_fmaf(qa[h].y, ka[k].y, s);
      s = __builtin_fmaf(qa[h].z, ka[k].z, s);
      s = __builtin_fmaf(qa[h].w, ka[k].w, s);
      s = __builtin_fmaf(qb[h].x, kb[k].x, s);
      s = __builtin_fmaf(qb[h].y, kb[k].y, s);
      s = __builtin_fmaf(qb[h].z, kb[k].z, s);
      s = __builtin_fmaf(qb[h].w, kb[k].w, s);
      s = LPP == 16 ? gq_row16_sum(s) : gq_row8_sum(s);
      if (sub == 0 && j < n) ss[h][j] = s * a.scale;
    }
  }
  __syncthreads();

  /* phase 2: chunk max, exponentials and their sum per head */
  const size_t ml = (size_t)a.nch * 2;
  for (int h = wave; h < G; h += kThreads / GQ_WAVE) {
    float m = -INFINITY;
    for (int j = lane; j < n; j += GQ_WAVE) m = fmaxf(m, ss[h][j]);
    m = gq_wave_max(m);
    float l = 0.f;
    for (int j = lane; j < n; j += GQ_WAVE) {
      const float e = expf(ss[h][j] - m);
      ss[h][j] = e;
      l += e;
    }
    l = gq_wave_sum(l);
    if (lane == 0) {
      gst<float>(a.part_ml + (size_t)(h0 + h) * ml + 2 * c, m);
      gst<float>(a.part_ml + (size_t)(h0 + h) * ml + 2 * c + 1, l);
    }
  }
  __syncthreads();

  /* phase 3: o = sum_j p_j V_j over the chunk */
  float4 acc[G];
#pragma unroll
  for (int h = 0; h < G; h++) acc[h] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < VIT; k++) {
    const int j = pg + NPG * k;
    if (j < n) {
#pragma unroll
      for (int h = 0; h < G; h++) {
        const float p = ss[h][j];
        acc[h].x = __builtin_fmaf(p, vr[k].x, acc[h].x);
        acc[h].y = __builtin_fmaf(p, vr[k].y, acc[h].y);
        acc[h].z = __builtin_fmaf(p, vr[k].z, acc[h].z);
        acc[h].w = __builtin_fmaf(p, vr[k].w, acc[h].w);
      }
    }
  }
#pragma unroll
  for (int h = 0; h < G; h++) sr[pg][h][dg] = acc[h];
  __syncthreads();
  for (int t = tid; t < G * DG; t += kThreads) {
    const int h = t / DG, q = t - h * DG;
    float4 o = sr[0][h][q];
#pragma unroll
    for (int p = 1; p < NPG; p++) {
      const float4 u = sr[p][h][q];
      o.x += u.x, o.y += u.y, o.z += u.z, o.w += u.w;
    }
    gst<float4>(a.part_o + ((size_t)(h0 + h) * a.nch + c) * HD + 4 * q, o);
  }
}

template <int HD, int G, int S>
__global__ __launch_bounds__(kThreads) void attn_partial_kernel(AttnArgs a) {
  attn_partial_body<HD, G, S>(a);
}

/* 32-position chunks at 7 waves per SIMD: 72 VGPRs, no spill (the free
 * allocation took 79, six waves).  The 2,056 workgroups of ctx 8193 then
 * take ~1.15 rounds instead of ~1.35: 18.9 against 19.1 us per layer, decode
 * +0.4%.  Eight waves (64 VGPRs) spilled and ran at 29.7 us. */
template <int HD, int G>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(7, 8))) void attn_partial32_kernel(AttnArgs a) {
  attn_partial_body<HD, G, 32>(a);
}

/* Dimensions of one query head per merge workgroup.  16 (256 workgroups at
 * 32 heads x 128) measured faster in the graph-replayed decode than 32:
 * each thread's chain of chunk loads is half as long. */
constexpr int kMergeDims = 16;

/* Merge the chunks of one query head for kMergeDims of its dimensions:
 * out = sum_c o_c e^(m_c - M) / sum_c l_c e^(m_c - M). */
__global__ __launch_bounds__(kThreads) void attn_merge_kernel(AttnArgs a) {
  constexpr int NG = kThreads / kMergeDims; /* chunk groups */
  extern __shared__ float sw[]; /* [nch] weights e^(m_c - M), then l_c */
  __shared__ float red[kThreads / GQ_WAVE];
  __shared__ float sacc[NG][kMergeDims];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int pos = a.pos_dev ? gld<int>(a.pos_dev) : a.pos;
  const int L = min(pos + 1, a.max_seq);
  const int nc = (L + a.s_max - 1) / a.s_max;
  const float *ml = a.part_ml + (size_t)h * a.nch * 2;
  float *sl = sw + a.nch;
  float m = -INFINITY;
  for (int c = tid; c < nc; c += kThreads) {
    const float mc = gld<float>(ml + 2 * c);
    sw[c] = mc;
    sl[c] = gld<float>(ml + 2 * c + 1);
    m = fmaxf(m, mc);
  }
  m = gq_wave_max(m);
  if (lane == 0) red[wave] = m;
  __syncthreads();
  const float M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float l = 0.f;
  for (int c = tid; c < nc; c += kThreads) {
    const float w = expf(sw[c] - M);
    sw[c] = w;
    l = __builtin_fmaf(sl[c], w, l);
  }
  l = gq_wave_sum(l);
  __syncthreads();
  if (lane == 0) red[wave] = l;
  __syncthreads();
  const float Ls = (red[0] + red[1]) + (red[2] + red[3]);
  const int d = blockIdx.y * kMergeDims + tid % kMergeDims, cg = tid / kMergeDims;
  const float *o = a.part_o + (size_t)h * a.nch * a.hd + d;
  float acc = 0.f;
  /* unrolled so a thread's ~16 chunk loads (260 chunks at ctx 8192 over 16
   * chunk groups) go out in one batch: decode +0.4% against unroll 8 */
#pragma unroll 16
  for (int c = cg; c < nc; c += NG) acc = __builtin_fmaf(gld<float>(o + (size_t)c * a.hd), sw[c], acc);
  sacc[cg][tid % kMergeDims] = acc;
  __syncthreads();
  if (tid < kMergeDims) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < NG; k++) t += sacc[k][tid];
    gst<float>(a.out + (size_t)h * a.hd + d, t / Ls);
  }
}

template <int HD, int G>
int launch_partial(const AttnArgs &a, hipStream_t s) {
  if (a.s_max == 128)
    hipLaunchKernelGGL((attn_partial_kernel<HD, G, 128>), dim3(a.n_kv, a.nch), dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((attn_partial32_kernel<HD, G>), dim3(a.n_kv, a.nch), dim3(kThreads), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}

} // namespace

int gq_attn_nch(int n_kv, int max_seq) {
  (void)n_kv;
  const int s = chunk_for(max_seq);
  return (max_seq + s - 1) / s;
}

int gq_attn_smax(int max_seq, int nch) {
  (void)nch;
  return chunk_for(max_seq);
}

int gq_launch_attention(const AttnArgs &a, hipStream_t s, hipEvent_t mid) {
  if (a.n_kv <= 0 || a.n_heads % a.n_kv || a.nch != gq_attn_nch(a.n_kv, a.max_seq) ||
      a.s_max != chunk_for(a.max_seq))
    return -1;
  if (a.hd % 32 || (size_t)a.nch * 2 * sizeof(float) > 32768) return -1;
  const int G = a.n_heads / a.n_kv;
  int rc = -1;
  if (a.hd == 128 && G == 4) rc = launch_partial<128, 4>(a, s);
  else if (a.hd == 128 && G == 8) rc = launch_partial<128, 8>(a, s);
  else if (a.hd == 128 && G == 1) rc = launch_partial<128, 1>(a, s);
  else if (a.hd == 128 && G == 2) rc = launch_partial<128, 2>(a, s);
  else if (a.hd == 64 && G == 4) rc = launch_partial<64, 4>(a, s);
  else if (a.hd == 64 && G == 8) rc = launch_partial<64, 8>(a, s);
  else if (a.hd == 64 && G == 1) rc = launch_partial<64, 1>(a, s);
  else if (a.hd == 64 && G == 2) rc = launch_partial<64, 2>(a, s);
  if (rc) return rc;
  if (mid) (void)hipEventRecord(mid, s);
  hipLaunchKernelGGL(attn_merge_kernel, dim3(a.n_heads, a.hd / kMergeDims), dim3(kThreads),
                     (size_t)a.nch * 2 * sizeof(float), s, a);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}

namespace {

typedef float gq_f32x4 __attribute__((ext_vector_type(4)));
typedef float gq_f2a __attribute__((ext_vector_type(2)));
typedef __bf16 gq_bf2a __attribute__((ext_vector_type(2)));

/* Causal attention of a prefill chunk on the fp32 matrix cores
 * (v_mfma_f32_16x16x4_f32), flash-attention style: one wave per 16 query
 * rows = 16 / G tokens x the G query heads of KV head g (the heads that
 * share K/V), streaming the keys 0 .. (last token's position) in blocks of
 * 16 with an online softmax.  Per block:
 *   S^T = K Q^T   D[key][row]: lane (c, j) = (lane % 16, lane / 16) holds
 *                 row c, keys 4 j + i (i < 4); the head dimension is split
 *                 into 4 lane groups (dims HD/4 j ..) so every MFMA step
 *                 reads one K and one Q float per lane;
 *   scale, mask keys past each row's position, running max / sum across
 *   the 4 lanes of a row;
 *   O += P V      A = P straight from the S^T layout (step i takes keys
 *                 4 j + i), B = V rows; output tile d holds dims ND c + d,
 *                 so a lane reads ND consecutive floats of each V row and
 *                 holds ND consecutive output dims of rows 4 j + i.
 * Four waves per workgroup take every fourth key block each and combine
 * their (max, sum, O) through LDS at the end, so the longest causal rows
 * finish in a quarter of the time.  One register buffer per wave: the next
 * block's K loads once the scores have read K, its V once P V has read V,
 * which keeps the kernel at 208 VGPRs, two waves per SIMD (two buffers
 * needed 312, one wave per SIMD, and ran 1.25-1.4x slower).  Same mathematics as the reference (engine.c:476-501:
 * scores * 1/sqrt(hd), -inf past the query position, softmax, P V) in fp32
 * throughout; only the summation order differs. */
template <int HD>
struct FlashLds { /* the waves' (max, sum, O) on their way to wave 0 */
  float xm[3][64], xl[3][64], xo[3][HD / 16 * 4][64];
};

template <int HD, int G>
__device__ __forceinline__ void flash_tile(const AttnArgs &a, int g, int t0, int wv, FlashLds<HD> &lds) {
  constexpr int TPT = 16 / G; /* tokens per tile */
  constexpr int NS = HD / 4;  /* QK^T MFMA steps */
  constexpr int ND = HD / 16; /* output tiles over the head dimension */
  auto &xm = lds.xm, &xl = lds.xl;
  auto &xo = lds.xo;
  const int lane = threadIdx.x & 63, c = lane & 15, j = lane >> 4;
  const int last = min(t0 + TPT, a.ntok) - 1;
  const int pmax = a.pos + last; /* last key any row of the tile needs */
  /* B operand of S^T: row c's query, dims NS j .. NS j + NS - 1 */
  const int qt = min(t0 + c / G, a.ntok - 1), qh = g * G + c % G;
  float qv[NS];
  {
    const float *qp = a.q + (size_t)qt * a.q_stride + (size_t)qh * HD + NS * j;
#pragma unroll
    for (int s4 = 0; s4 < NS / 4; s4++) {
      const float4 v = gld<float4>(qp + 4 * s4);
      qv[4 * s4] = v.x, qv[4 * s4 + 1] = v.y, qv[4 * s4 + 2] = v.z, qv[4 * s4 + 3] = v.w;
    }
  }
  const int cpos = a.pos + t0 + c / G; /* row c's position (S^T layout) */
  const float *K = a.k + (size_t)g * a.max_seq * HD;
  const float *V = a.v + (size_t)g * a.max_seq * HD;
  float m = -INFINITY, l = 0.f;
  gq_f32x4 o[ND];
#pragma unroll
  for (int d = 0; d < ND; d++) o[d] = gq_f32x4{0.f, 0.f, 0.f, 0.f};
  const int nblk = pmax / 16 + 1;
  /* K row key0 + c, dims NS j ..; V rows key0 + 4 j + i, dims ND c ..
   * (rows past pmax are never weighted: zeroed so stale cache contents
   * cannot leak in as 0 * inf). */
  float kv[NS], vv[4][ND];
  auto loadk = [&](int key0, float (&kq)[NS]) {
    const float *kp = K + (size_t)min(key0 + c, a.max_seq - 1) * HD + NS * j;
#pragma unroll
    for (int s4 = 0; s4 < NS / 4; s4++) {
      const float4 v = gld<float4>(kp + 4 * s4);
      kq[4 * s4] = v.x, kq[4 * s4 + 1] = v.y, kq[4 * s4 + 2] = v.z, kq[4 * s4 + 3] = v.w;
    }
  };
  auto loadv = [&](int key0, float (&vq)[4][ND]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int key = key0 + 4 * j + i;
      const float *vp = V + (size_t)min(key, a.max_seq - 1) * HD + ND * c;
#pragma unroll
      for (int d4 = 0; d4 < ND / 4; d4++) {
        float4 v = gld<float4>(vp + 4 * d4);
        if (key > pmax) v = make_float4(0.f, 0.f, 0.f, 0.f);
        vq[i][4 * d4] = v.x, vq[i][4 * d4 + 1] = v.y, vq[i][4 * d4 + 2] = v.z, vq[i][4 * d4 + 3] = v.w;
      }
    }
  };
  /* one key block: S^T (four independent MFMA chains), mask, online
   * softmax, rescale, O += P V */
  auto stepS = [&](int key0, const float (&kq)[NS], float (&p)[4]) {
    gq_f32x4 sp[4];
#pragma unroll
    for (int u = 0; u < 4; u++) sp[u] = gq_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s++) sp[s & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(kq[s], qv[s], sp[s & 3], 0, 0, 0);
    const gq_f32x4 st = (sp[0] + sp[1]) + (sp[2] + sp[3]);
    /* st[i] = q(row c) . k(key0 + 4 j + i) */
    float sv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sv[i] = key0 + 4 * j + i <= cpos ? st[i] * a.scale : -INFINITY;
    float mb = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
    mb = fmaxf(mb, __shfl_xor(mb, 16, 64));
    mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
    /* a wave's rows may not see any key of its first blocks (the second
     * wave starts at block 1): keep m = -inf and weigh those blocks 0 */
    const float mn = fmaxf(m, mb);
    const float ms = mn == -INFINITY ? 0.f : mn;
    const float alpha = __expf(m - ms);
    float lb = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      p[i] = __expf(sv[i] - ms);
      lb += p[i];
    }
    lb += __shfl_xor(lb, 16, 64);
    lb += __shfl_xor(lb, 32, 64);
    l = __builtin_fmaf(l, alpha, lb);
    m = mn;
    /* O rows 4 j + i take the rescale of row 4 j + i (held by lane 4 j + i) */
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float al = __shfl(alpha, 4 * j + i, 64);
#pragma unroll
      for (int d = 0; d < ND; d++) o[d][i] *= al;
    }
  };
  auto stepPV = [&](const float (&p)[4], const float (&vq)[4][ND]) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int d = 0; d < ND; d++) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i], vq[i][d], o[d], 0, 0, 0);
  };
  /* wave wv takes blocks wv, wv + 4, ...; the wave's next block loads into
   * the registers as the current one frees them */
  if (wv < nblk) loadk(16 * wv, kv), loadv(16 * wv, vv);
  for (int b = wv; b < nblk; b += 4) {
    float p[4];
    stepS(16 * b, kv, p);
    if (b + 4 < nblk) loadk(16 * (b + 4), kv);
    stepPV(p, vv);
    if (b + 4 < nblk) loadv(16 * (b + 4), vv);
  }
  /* combine: waves 1-3 hand (m, l, O) to wave 0 (wave 0 holds block 0, so
   * its m is finite; a wave that had no block has m = -inf and weighs 0) */
  if (wv > 0) {
    xm[wv - 1][lane] = m, xl[wv - 1][lane] = l;
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
      for (int i = 0; i < 4; i++) xo[wv - 1][4 * d + i][lane] = o[d][i];
  }
  __syncthreads();
  if (wv > 0) return;
#pragma unroll
  for (int w = 0; w < 3; w++) {
    const float m1 = xm[w][lane], mt = fmaxf(m, m1);
    const float s0 = __expf(m - mt), s1 = __expf(m1 - mt);
    l = l * s0 + xl[w][lane] * s1;
    m = mt;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float a0 = __shfl(s0, 4 * j + i, 64), a1 = __shfl(s1, 4 * j + i, 64);
#pragma unroll
      for (int d = 0; d < ND; d++) o[d][i] = o[d][i] * a0 + xo[w][4 * d + i][lane] * a1;
    }
  }
  /* out[row] = O[row] / l[row]; row 4 j + i -> token t0 + row / G, head
   * g G + row % G */
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = 4 * j + i, t = t0 + row / G, h = g * G + row % G;
    const float inv = 1.0f / __shfl(l, row, 64);
    if (t < a.ntok) {
      const size_t base = (size_t)t * a.out_stride + (size_t)h * HD + ND * c;
#pragma unroll
      for (int d4 = 0; d4 < ND / 4; d4++) {
        const float4 v = make_float4(o[4 * d4][i] * inv, o[4 * d4 + 1][i] * inv, o[4 * d4 + 2][i] * inv,
                                     o[4 * d4 + 3][i] * inv);
        if (a.out16) {
          uint2 u;
          u.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){v.x, v.y}, gq_bf2a));
          u.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){v.z, v.w}, gq_bf2a));
          gst<uint2>(a.out16 + base + 4 * d4, u);
        } else {
          gst<float4>(a.out + base + 4 * d4, v);
        }
      }
    }
  }
}

/* One linear grid: workgroup L runs on XCD L mod 8, and takes KV head
 * L mod n_kv, so a head's K/V stays in one XCD's L2 (n_kv = 8: one head
 * per XCD; with tile-major ids every XCD read every head's K/V, 4 MB at
 * 512 tokens: 49.3 -> 38.6 us per layer).  Heavy (late) tiles first. */
template <int HD, int G>
__global__ __launch_bounds__(256) void flash_prefill_kernel(AttnArgs a) {
  __shared__ FlashLds<HD> lds;
  const int ntile = gridDim.x / a.n_kv;
  const int g = blockIdx.x % a.n_kv, tile = ntile - 1 - blockIdx.x / a.n_kv;
  flash_tile<HD, G>(a, g, tile * (16 / G), __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lds);
}

/* The same attention on the bf16 matrix cores without giving up fp32: every
 * fp32 operand x is the sum of three bf16 numbers, hi = bf16(x), mid =
 * bf16(x - hi), lo = bf16(x - hi - mid) (8 + 8 + 8 bits of a 24-bit
 * significand), and a product keeps the six of the nine partial products that
 * are not below 2^-24 of it: hi hi + (hi mid + mid hi) + (hi lo + lo hi + mid
 * mid), each exact, summed in fp32.  bf16 products run 16 times as fast as
 * fp32 ones (v_mfma_f32_16x16x4_f32), so six of them cost 0.38 of one.
 *
 * One workgroup of eight waves takes 128 query rows = 128 / G tokens x the
 * G query heads of a KV head, and streams the keys in blocks of 64: wave (rg,
 * kh) rows 32 rg .. + 31 against keys 32 kh .. + 31 of every block, online
 * softmax, the two halves of the keys combined at the end.  K and V are
 * loaded once per workgroup a block ahead into registers, split, and put into
 * LDS as three bf16 planes each (96 KB at head_dim 128):
 *   S^T = K Q^T   A = K planes [key][dim], B = Q planes, in registers for the
 *                 whole kernel; lane (r, h) = (lane % 32, lane / 32) gets row
 *                 r's scores of keys 8 a + 4 h + c (a, c < 4)
 *   O^T += V^T P^T  B = the probabilities straight from that layout: the 16
 *                 keys of a step are taken in the order in which a lane holds
 *                 them, and V is stored [dim][key] in the same order; lane
 *                 (r, h) holds row r's output dims, so the softmax's rescale
 *                 and the final division need no exchange between lanes.
 * Octets (8 bf16, 16 bytes) are XOR-swizzled by the row, so operand reads
 * are free of bank conflicts.
 *
 * Launches that would leave CUs idle split the keys over the grid
 * (AttnArgs.fs_split): each part leaves its unnormalised O, maximum and sum
 * to flash_merge_kernel.
 *
 * Microseconds with RoPE and append, 32 heads over 8, head_dim 128, beside
 * the fp32 kernel's: 512 tokens at 3584 379 -> 211 (two parts; 270 with 64
 * rows a workgroup), 2048 at 0 429 -> 239, 128 at 2000 71 -> 56, 37 at 8000
 * 244 -> 109 (both with the keys in parts).  The error against float64 of the
 * first is 6e-7 -> 2.5e-7.  Bound by what comes between the matrix
 * instructions, 192 of 32 cycles a SIMD or 2.6 of a block's 6.1 us: splitting
 * 32 values and 16 probabilities a lane, the exponentials, 56 KB of operands a
 * wave from LDS.  256 VGPRs at two waves per SIMD; at head_dim 128 they do
 * not hold everything, 19 to 22 values a lane spill (64-76 bytes of scratch).
 *
 * An infinity or NaN among the operands leaves NaN in the splits and so in
 * the outputs it reaches; a tile with an output that is not finite is computed
 * again by flash_tile, which treats them as fp32 arithmetic does. */
typedef __bf16 gq_bf8a __attribute__((ext_vector_type(8)));
typedef float gq_f16a __attribute__((ext_vector_type(16)));

constexpr int kFsKeys = 64, kFsRows = 128, kFsThreads = 512;

/* The launch for ntok tokens at pos: the fp32 kernel (split 0), or the
 * split-bf16 kernel with its keys in so many parts, whichever should take
 * less.  A 64-key block takes a workgroup of the fp32 kernel longer the more of
 * them share a CU; one CU runs one of the other kernel at a time, and its
 * partial O cross memory where the keys are split.  The tiles of a causal
 * prompt are of all lengths and fill each other's rounds, but for what the
 * last round leaves idle.
 *
 * The constants, microseconds, are fitted to 4410 launches timed with every
 * choice (fifteen head geometries at head_dim 64 and 128, 8 to 2048 tokens at 0
 * to 7500): the rule's choices take 0.7% more than the best ones, 11% more for
 * the worst in a hundred, and at most 6% more than the fp32 kernel.  The rule
 * before it (half the time at head_dim 64, causal tiles that fill every round)
 * took 75 of them to a slower kernel: 900 tokens of 8 heads at 0, head_dim 128,
 * 61 us in five parts against 48. */
struct FlashShape {
  int split, wgs;
};
constexpr int kFsMaxSplit = 8;
FlashShape flash_shape(int ntok, int pos, int n_heads, int n_kv, int hd, int n_cu, bool parts) {
  const int G = n_heads / n_kv, tpt = kFsRows / G, wgs = (ntok + tpt - 1) / tpt * n_kv;
  const int nblk = (pos + ntok - 1) / kFsKeys + 1; /* the longest tile's */
  const double mean = (pos + 0.5 * ntok) / kFsKeys + 1;
  const double even = (double)pos / (pos + ntok), causal = 1 - even; /* how far the tiles are of one length, and not */
  const bool wide = hd > 64;
  const double w = (double)((ntok + 16 / G - 1) / (16 / G)) * n_kv / n_cu; /* fp32 workgroups a CU */
  const double few = w <= 1 ? (wide ? 1.35 : 1.2) : (wide ? 2.45 : 1.6), many = wide ? 1.38 : 0.84;
  double best = w <= 2 ? few * nblk
                       : even * (nblk + mean) / 2 * many * std::max(w, std::min(std::ceil(w), 3.0)) +
                             causal * std::max(few * nblk, 1.25 * many * w * mean);
  FlashShape f{0, wgs};
  for (int k = 1; k == 1 || (parts && k <= kFsMaxSplit && nblk / k >= 2); k++) {
    const double r = (double)wgs * k / n_cu;
    const double blocks =
        r <= 1 ? nblk : std::max((double)nblk, even * std::ceil(r) * mean + causal * (r * mean + 0.3 * nblk));
    const double us = (wide ? 6.06 : 3.72) * blocks / k + (r > 1 ? 3.7 * causal : 0.0) +
                      (k > 1 ? 4.4 + 12.5 * k * ntok * n_heads * hd / 4.0e6 : 0.0);
    if (us < best) best = us, f.split = k;
  }
  return f;
}

/* two floats to their (hi, mid, lo) bf16 pairs, each rounded to nearest even */
__device__ __forceinline__ void split3(float x, float y, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){x, y}, gq_bf2a));
  x -= __builtin_bit_cast(float, hi << 16), y -= __builtin_bit_cast(float, hi & 0xffff0000u);
  mid = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){x, y}, gq_bf2a));
  x -= __builtin_bit_cast(float, mid << 16), y -= __builtin_bit_cast(float, mid & 0xffff0000u);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){x, y}, gq_bf2a));
}

/* four consecutive outputs, fp32 or bf16 */
__device__ __forceinline__ void flash_store(const AttnArgs &a, size_t at, const float (&y)[4]) {
  if (a.out16) {
    uint2 u;
    u.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){y[0], y[1]}, gq_bf2a));
    u.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2a){y[2], y[3]}, gq_bf2a));
    gst<uint2>(a.out16 + at, u);
  } else {
    gst<float4>(a.out + at, make_float4(y[0], y[1], y[2], y[3]));
  }
}

struct Split8 {
  uint4 p[3];
};
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  Split8 s;
  split3(x[0], x[1], s.p[0].x, s.p[1].x, s.p[2].x);
  split3(x[2], x[3], s.p[0].y, s.p[1].y, s.p[2].y);
  split3(x[4], x[5], s.p[0].z, s.p[1].z, s.p[2].z);
  split3(x[6], x[7], s.p[0].w, s.p[1].w, s.p[2].w);
  return s;
}

/* the pairs of planes whose product is kept: the small ones, and last hi hi */
constexpr int kFsA[6] = {1, 2, 0, 1, 0, 0}, kFsB[6] = {1, 0, 2, 0, 1, 0};

template <int HD, int G>
__global__ __launch_bounds__(kFsThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void flash_split_kernel(AttnArgs a) {
  constexpr int TPT = kFsRows / G;       /* tokens per workgroup */
  constexpr int NO = HD / 8;             /* octets of a K row */
  constexpr int NSL = HD / 16;           /* dim slices of S^T */
  constexpr int ND = HD / 32;            /* dim tiles of O^T */
  constexpr int KPL = kFsKeys * HD * 2;  /* bytes of one K (or V) plane */
  constexpr int KT = kFsKeys * NO / kFsThreads; /* K octets per thread */
  constexpr int VTH = kFsKeys / 8 * HD / 2; /* threads with a V task: 8 keys x 2 dims */
  static_assert(6 * KPL >= 2 * (int)sizeof(FlashLds<HD>) && 6 * KPL >= 4 * 64 * 4 * (ND * 16 + 2), "exchanges fit the planes");
  /* K's planes, V's planes, and Q's third plane [slice][row group][lane]: in
   * registers it did not fit beside the other two */
  __shared__ __attribute__((aligned(16))) uint8_t smem_[6 * KPL + NSL * 4096];
  __shared__ int s_bad;
  GQ_LDS uint8_t *smem = (GQ_LDS uint8_t *)smem_;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), rg = wv >> 1, kh = wv & 1;
  /* heads and tiles as in flash_prefill_kernel */
  const int ntile = gridDim.x / a.n_kv;
  const int g = blockIdx.x % a.n_kv, tile = ntile - 1 - blockIdx.x / a.n_kv, t0 = tile * TPT;
  const int pmax = a.pos + min(t0 + TPT, a.ntok) - 1; /* last key any row of the tile needs */
  const int nblk = pmax / kFsKeys + 1;
  /* this part's key blocks b0 .. b1 - 1 */
  const int b0 = nblk * (int)blockIdx.y / a.fs_split, b1 = nblk * ((int)blockIdx.y + 1) / a.fs_split;
  const float *K = a.k + (size_t)g * a.max_seq * HD;
  const float *V = a.v + (size_t)g * a.max_seq * HD;
  if (tid == 0) s_bad = 0;
  /* this lane's query row: token t0 + row / G, head g G + row % G */
  const int row = 32 * rg + r, qt = min(t0 + row / G, a.ntok - 1), qh = g * G + row % G;
  const int cpos = a.pos + t0 + row / G;
  uint4 q[NSL][2]; /* dims 16 s + 8 h .. + 7 */
  const uint32_t qlo = (uint32_t)(6 * KPL + (rg * 64 + lane) * 16);
#pragma unroll
  for (int s = 0; s < NSL; s++) {
    const float *qp = a.q + (size_t)qt * a.q_stride + (size_t)qh * HD + 16 * s + 8 * h;
    const float4 u = gld<float4>(qp), v = gld<float4>(qp + 4);
    const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    const Split8 p = split8(x);
    q[s][0] = p.p[0], q[s][1] = p.p[1];
    if (kh == 0) lst<uint4>(smem, qlo + 4096 * s, p.p[2]);
  }
  /* K tasks: octet ko of keys tid / NO + (512 / NO) i; V task: dims 2 vd ..
   * of the eight keys of octet vo, in P's order: key octet 4 kh + 2 t + h is
   * keys 32 kh + 16 t + 4 h + {0..3, 8..11} */
  const int ko = tid % NO, kk = tid / NO;
  const int vd = tid % (HD / 2), vo = (tid / (HD / 2)) & 7;
  const int vkey = 32 * (vo >> 2) + 16 * ((vo >> 1) & 1) + 4 * (vo & 1);
  float4 kr[KT][2];
  float2 vr[8];
  auto load = [&](int b) {
    const int key0 = b * kFsKeys;
#pragma unroll
    for (int i = 0; i < KT; i++) {
      const float *kp = K + (size_t)min(key0 + kk + kFsThreads / NO * i, pmax) * HD + 8 * ko;
      kr[i][0] = gld<float4>(kp), kr[i][1] = gld<float4>(kp + 4);
    }
    if (VTH == kFsThreads || tid < VTH) {
#pragma unroll
      for (int e = 0; e < 8; e++) /* keys past pmax repeat it: their weight is 0 */
        vr[e] = gld<float2>(V + (size_t)min(key0 + vkey + (e & 3) + 8 * (e >> 2), pmax) * HD + 2 * vd);
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < KT; i++) {
      const float x[8] = {kr[i][0].x, kr[i][0].y, kr[i][0].z, kr[i][0].w, kr[i][1].x, kr[i][1].y, kr[i][1].z, kr[i][1].w};
      const Split8 s = split8(x);
      const int key = kk + kFsThreads / NO * i;
      const uint32_t at = (uint32_t)(key * HD * 2 + ((ko ^ (key & (NO - 1))) << 4));
#pragma unroll
      for (int p = 0; p < 3; p++) lst<uint4>(smem, (uint32_t)(p * KPL) + at, s.p[p]);
    }
    if (VTH == kFsThreads || tid < VTH) {
#pragma unroll
      for (int d = 0; d < 2; d++) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = d == 0 ? vr[e].x : vr[e].y;
        const Split8 s = split8(x);
        const int dim = 2 * vd + d;
        const uint32_t at = (uint32_t)(3 * KPL + dim * kFsKeys * 2 + ((vo ^ ((dim ^ (dim >> 3)) & 7)) << 4));
#pragma unroll
        for (int p = 0; p < 3; p++) lst<uint4>(smem, (uint32_t)(p * KPL) + at, s.p[p]);
      }
    }
  };
  /* operand addresses: K row 32 kh + r, octet 2 s + h; V row 32 d + r, octet
   * 4 kh + 2 t + h */
  const int krow = 32 * kh + r;
  const uint32_t kbase = (uint32_t)(krow * HD * 2 + ((h ^ (krow & (NO - 1))) << 4));
  const uint32_t vbase = (uint32_t)(r * kFsKeys * 2 + (((4 * kh + h) ^ ((r ^ (r >> 3)) & 7)) << 4));
  float m = -INFINITY, l = 0.f;
  gq_f16a o[ND];
#pragma unroll
  for (int d = 0; d < ND; d++) o[d] = gq_f16a{};
  if (b0 < b1) load(b0);
  for (int b = b0; b < b1; b++) {
    __syncthreads(); /* the planes are free */
    stage();
    __syncthreads();
    if (b + 1 < b1) load(b + 1);
    const int key0 = b * kFsKeys + 32 * kh;
    if (key0 > pmax) continue; /* none of this wave's keys (uniform in the wave) */
    /* addresses from these, one XOR each, anew in every block: kept across
     * blocks they cost the registers that O needs */
    uint32_t kb = kbase, vb = vbase, qb = qlo;
    asm volatile("" : "+v"(kb), "+v"(vb), "+v"(qb));
    gq_f16a sa = gq_f16a{}, sb = gq_f16a{};
#pragma unroll
    for (int s = 0; s < NSL; s++) {
      gq_bf8a kv[3];
      const gq_bf8a qv[3] = {__builtin_bit_cast(gq_bf8a, q[s][0]), __builtin_bit_cast(gq_bf8a, q[s][1]),
                             lld<gq_bf8a>(smem, qb + 4096 * s)};
#pragma unroll
      for (int p = 0; p < 3; p++)
        kv[p] = lld<gq_bf8a>(smem, (kb ^ (32 * s)) + p * KPL);
#pragma unroll
      for (int u = 0; u < 6; u++) {
        if (u < 5) sb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kv[kFsA[u]], qv[kFsB[u]], sb, 0, 0, 0);
        else sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kv[kFsA[u]], qv[kFsB[u]], sa, 0, 0, 0);
      }
    }
    /* scores of keys key0 + 8 (e / 4) + 4 h + e % 4 */
    float p[16], mb = -INFINITY;
    if (key0 + 31 <= a.pos + t0) { /* every row sees every key of this half block */
#pragma unroll
      for (int e = 0; e < 16; e++) p[e] = (sa[e] + sb[e]) * a.scale;
    } else {
#pragma unroll
      for (int e = 0; e < 16; e++)
        p[e] = key0 + 8 * (e >> 2) + 4 * h + (e & 3) <= cpos ? (sa[e] + sb[e]) * a.scale : -INFINITY;
    }
#pragma unroll
    for (int e = 0; e < 16; e++) mb = fmaxf(mb, p[e]);
    mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
    /* a half may hold no visible key of a row yet: m stays -inf, weight 0 */
    const float mn = fmaxf(m, mb), ms = mn == -INFINITY ? 0.f : mn;
    const float alpha = __expf(m - ms);
    float lb = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      p[e] = __expf(p[e] - ms);
      lb += p[e];
    }
    lb += __shfl_xor(lb, 32, 64);
    l = __builtin_fmaf(l, alpha, lb);
    m = mn;
    Split8 ps[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; e++) x[e] = p[8 * t + e];
      ps[t] = split8(x);
    }
    /* the half block's P V in accumulators of its own: O takes one rounding
     * per 32 keys (twelve with O itself as the accumulator, and the error
     * over 4096 keys was above the fp32 kernel's) */
#pragma unroll
    for (int d = 0; d < ND; d++) {
      if (HD > 64) __builtin_amdgcn_sched_barrier(0); /* no operands read further ahead: registers */
      gq_f16a pv = gq_f16a{};
#pragma unroll
      for (int t = 0; t < 2; t++) {
        gq_bf8a vv[3];
#pragma unroll
        for (int q3 = 0; q3 < 3; q3++)
          vv[q3] = lld<gq_bf8a>(smem, (vb ^ (((4 * d & 7) ^ (2 * t)) << 4)) + (3 + q3) * KPL + 32 * d * kFsKeys * 2);
#pragma unroll
        for (int u = 0; u < 6; u++)
          pv = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv[kFsA[u]], __builtin_bit_cast(gq_bf8a, ps[t].p[kFsB[u]]), pv, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 16; e++) o[d][e] = __builtin_fmaf(o[d][e], alpha, pv[e]);
    }
  }
  /* the two halves of the keys: kh = 1 hands (m, l, O) to kh = 0 */
  __syncthreads();
  GQ_LDS float *x = (GQ_LDS float *)smem + rg * 64 * (ND * 16 + 2);
  if (kh == 1) {
    x[lane] = m, x[64 + lane] = l;
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
      for (int e = 0; e < 16; e++) x[64 * (2 + 16 * d + e) + lane] = o[d][e];
  }
  __syncthreads();
  if (kh == 0) {
    /* a half (or a whole part of the keys) that holds no visible key of a
     * row weighs 0; of an unsplit launch kh = 0 holds key 0 */
    const float m1 = x[lane], mt = fmaxf(m, m1), mf = mt == -INFINITY ? 0.f : mt;
    const float s0 = __expf(m - mf), s1 = __expf(m1 - mf), lt = l * s0 + x[64 + lane] * s1;
    const bool parts = a.fs_split > 1;
    const float inv = parts ? 1.0f : 1.0f / lt;
    const int t = t0 + row / G;
    bool bad = false;
    float *po = a.part_o + ((size_t)blockIdx.y * a.ntok + t) * (a.n_heads * HD) + qh * HD;
    if (parts && t < a.ntok && h == 0) {
      float *ml = a.part_ml + (((size_t)blockIdx.y * a.ntok + t) * a.n_heads + qh) * 2;
      ml[0] = mt, ml[1] = lt;
    }
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
      for (int c = 0; c < 4; c++) { /* dims 32 d + 8 c + 4 h .. + 3 */
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          y[e] = (o[d][4 * c + e] * s0 + x[64 * (2 + 16 * d + 4 * c + e) + lane] * s1) * inv;
          bad |= !(__builtin_fabsf(y[e]) < INFINITY);
        }
        const int dim = 32 * d + 8 * c + 4 * h;
        if (t < a.ntok) {
          const size_t at = (size_t)t * a.out_stride + (size_t)qh * HD + dim;
          if (parts) gst<float4>(po + dim, make_float4(y[0], y[1], y[2], y[3]));
          else flash_store(a, at, y);
        }
      }
    if (!parts && __ballot(bad) && lane == 0) s_bad = 1;
  }
  __syncthreads();
  if (!s_bad) return;
  /* two 16-row tiles at a time, four waves each */
  for (int t = t0; t < min(t0 + TPT, a.ntok); t += 32 / G) {
    flash_tile<HD, G>(a, g, min(t + (wv >> 2) * (16 / G), (a.ntok - 1) / (16 / G) * (16 / G)), wv & 3, ((FlashLds<HD> *)smem_)[wv >> 2]);
    __syncthreads();
  }
}

/* The parts of a key-split launch: out = sum_s O_s e^(m_s - M) / sum_s l_s
 * e^(m_s - M), a workgroup per 16 query rows (16 / G tokens x G heads),
 * sixteen lanes a row; a tile with a result that is not finite goes through
 * flash_tile. */
template <int HD, int G>
__global__ __launch_bounds__(256) void flash_merge_kernel(AttnArgs a) {
  __shared__ FlashLds<HD> lds;
  __shared__ int s_bad;
  const int ntile = gridDim.x / a.n_kv;
  const int g = blockIdx.x % a.n_kv, tile = ntile - 1 - blockIdx.x / a.n_kv, t0 = tile * (16 / G);
  const int row = threadIdx.x >> 4, sub = threadIdx.x & 15, t = t0 + row / G, qh = g * G + row % G;
  if (threadIdx.x == 0) s_bad = 0;
  __syncthreads();
  if (t < a.ntok) {
    const float *ml = a.part_ml + ((size_t)t * a.n_heads + qh) * 2, *po = a.part_o + (size_t)t * (a.n_heads * HD) + qh * HD;
    const size_t mls = (size_t)a.ntok * a.n_heads * 2, pos = (size_t)a.ntok * a.n_heads * HD;
    float M = -INFINITY, L = 0.f;
    for (int s = 0; s < a.fs_split; s++) M = fmaxf(M, ml[s * mls]);
    for (int s = 0; s < a.fs_split; s++) L += ml[s * mls + 1] * __expf(ml[s * mls] - M);
    const float inv = 1.0f / L;
    bool bad = false;
#pragma unroll
    for (int d = 0; d < HD / 64; d++) {
      const int dim = 64 * d + 4 * sub;
      float y[4] = {0.f, 0.f, 0.f, 0.f};
      for (int s = 0; s < a.fs_split; s++) {
        const float w = __expf(ml[s * mls] - M);
        const float4 u = gld<float4>(po + s * pos + dim);
        y[0] = __builtin_fmaf(u.x, w, y[0]), y[1] = __builtin_fmaf(u.y, w, y[1]);
        y[2] = __builtin_fmaf(u.z, w, y[2]), y[3] = __builtin_fmaf(u.w, w, y[3]);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) y[e] *= inv, bad |= !(__builtin_fabsf(y[e]) < INFINITY);
      flash_store(a, (size_t)t * a.out_stride + (size_t)qh * HD + dim, y);
    }
    if (bad) s_bad = 1;
  }
  __syncthreads();
  if (s_bad) flash_tile<HD, G>(a, g, t0, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lds);
}

template <int HD, int G>
int launch_flash(const AttnArgs &a0, int n_cu, hipStream_t s) {
  AttnArgs a = a0;
  const FlashShape f = flash_shape(a.ntok, a.pos, a.n_heads, a.n_kv, HD, n_cu, a.part_o != nullptr);
  a.fs_split = f.split;
  const int narrow = (a.ntok + 16 / G - 1) / (16 / G) * a.n_kv;
  if (!f.split) {
    hipLaunchKernelGGL((flash_prefill_kernel<HD, G>), dim3(narrow), dim3(256), 0, s, a);
  } else {
    hipLaunchKernelGGL((flash_split_kernel<HD, G>), dim3(f.wgs, f.split), dim3(kFsThreads), 0, s, a);
    if (f.split > 1) hipLaunchKernelGGL((flash_merge_kernel<HD, G>), dim3(narrow), dim3(256), 0, s, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -4;
}

} // namespace

bool gq_flash_takes(int n_heads, int n_kv, int hd) {
  if (n_kv <= 0 || n_heads <= 0 || n_heads % n_kv || (hd != 64 && hd != 128)) return false;
  const int G = n_heads / n_kv;
  return G == 1 || G == 2 || G == 4 || G == 8;
}

size_t gq_flash_parts(int ntok, int pos, int n_heads, int n_kv, int hd, int n_cu) {
  if (!gq_flash_takes(n_heads, n_kv, hd)) return 0; /* flash_shape divides by 16 / G */
  const FlashShape f = flash_shape(ntok, pos, n_heads, n_kv, hd, n_cu, true);
  return f.split > 1 ? (size_t)f.split * ntok * n_heads : 0;
}

int gq_launch_flash_prefill(const AttnArgs &a, int n_cu, hipStream_t s) {
  if (!gq_flash_takes(a.n_heads, a.n_kv, a.hd) || a.ntok < 1 || a.pos < 0 || a.pos + a.ntok > a.max_seq) return -1;
  const int G = a.n_heads / a.n_kv;
  if (a.hd == 128 && G == 4) return launch_flash<128, 4>(a, n_cu, s);
  if (a.hd == 128 && G == 8) return launch_flash<128, 8>(a, n_cu, s);
  if (a.hd == 128 && G == 1) return launch_flash<128, 1>(a, n_cu, s);
  if (a.hd == 128 && G == 2) return launch_flash<128, 2>(a, n_cu, s);
  if (a.hd == 64 && G == 4) return launch_flash<64, 4>(a, n_cu, s);
  if (a.hd == 64 && G == 8) return launch_flash<64, 8>(a, n_cu, s);
  if (a.hd == 64 && G == 1) return launch_flash<64, 1>(a, n_cu, s);
  if (a.hd == 64 && G == 2) return launch_flash<64, 2>(a, n_cu, s);
  return -1;
}

int gq_launch_rope_append(const RopeArgs &a, hipStream_t s) {
  if ((a.hd & 1) || a.n_kv <= 0 || a.n_heads % a.n_kv || a.ntok < 0 || (a.parts && a.kparts < 1)) return -1;
  hipLaunchKernelGGL(rope_append_kernel, dim3(std::max(a.ntok, 1) * a.n_kv), dim3(kThreads), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}
