/*
 * gq_dense.hip — the prefill GEMM of long prompts: bf16 activations against
 * bf16 weights on the matrix cores of gfx950, fp32 accumulation.
 *
 * pgemm_kernel (gq_prefill.hip) dequantizes K-quant blocks as it multiplies:
 * once per 128 tokens and weight, about as many vector-ALU cycles as its
 * MFMAs take.  That is right for few tokens, where the quantized bytes are
 * what there is to read; for many tokens the same weights are converted over
 * and over.  The first prompt of enough tokens therefore makes a bf16 copy
 * of the projections beside the quantized ones (2 bytes a weight, the values
 * that pgemm_kernel rounds to), and such prompts multiply by that.
 *
 * The copy is laid out as the kernel's LDS tiles: for each 256-row tile and
 * 32-column step one contiguous 16 KB block, row r's four octets (8 weights,
 * 16 bytes) at 64 r + 16 (o ^ ((r / 2) % 4)), so the weights stream in by
 * whole 1 KB DMA instructions and every MFMA operand is a ds_read_b128 free
 * of bank conflicts.  Gate and up share one copy, 32 rows of each in turn,
 * which puts a row's gate and up sums into the same lanes.
 *
 * Measured at the 8B shape, us per layer (quantized kernels / here): 512
 * tokens: q/k/v 50 / 45, o 33 / 29, gate + up 151 / 124, down 96 / 74; 1500
 * tokens in one chunk: 152 / 110, 103 / 70, 441 / 374, 344 / 191.  A
 * 1500-token prompt 38.3 -> 32.1 ms (40.8 in chunks of 512 before).  At 1500
 * tokens that is 0.69, 0.72, 0.94 and 0.92 PFLOP/s of the 1.45 that a large
 * library product reaches on the card: 144, 192, 672 and 192 workgroups leave
 * 44, 25, 12 and 25% of the 256 CUs idle, and one wave per SIMD waits at every
 * step's barrier.
 */
#include <algorithm>

#include "gq_device.h"
#include "gq_internal.h"

namespace {

typedef __bf16 gq_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gq_f32x16 __attribute__((ext_vector_type(16)));
typedef float gq_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 gq_bf2 __attribute__((ext_vector_type(2)));

constexpr int kDN = 256, kDK = 32;
constexpr int kDWStep = kDN * kDK * 2; /* bytes of a weight tile's step */

/* ---- the copy ---------------------------------------------------------- */
/* eight bf16 of eight fp32 weights, each the value that PW<>::dequant rounds */
__device__ __forceinline__ void put_octet(uint8_t *out, const float (&w)[8]) {
  uint32_t p[4];
#pragma unroll
  for (int i = 0; i < 4; i++) p[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((gq_f2){w[2 * i], w[2 * i + 1]}, gq_bf2));
  gst<uint4>(out, make_uint4(p[0], p[1], p[2], p[3]));
}

__device__ __forceinline__ uint32_t byte8(const uint2 &q, int i) { return ((i < 4 ? q.x : q.y) >> (8 * (i & 3))) & 0xffu; }

/* eight bytes from a 2-byte boundary */
__device__ __forceinline__ uint2 ld8(const uint8_t *p) {
  uint2 q;
  q.x = gld<uint16_t>(p) | ((uint32_t)gld<uint16_t>(p + 2) << 16);
  q.y = gld<uint16_t>(p + 4) | ((uint32_t)gld<uint16_t>(p + 6) << 16);
  return q;
}

/* Octet oct of each of a 256-column block's eight 32-column steps (Q8_0: of
 * eight blocks), step st to out + st * kDWStep: a lane reads its bytes of the
 * block once for all the steps that share them. */
__device__ __forceinline__ void octets_q4k(uint8_t *out, const uint8_t *b, int oct) {
  const uint4 h = gld<uint4>(b); /* d, dmin, the twelve bytes of scales and mins */
  const float d = gq_h2f(h.x & 0xffffu), dm = gq_h2f(h.x >> 16);
  uint2 q[4];
#pragma unroll
  for (int c = 0; c < 4; c++) q[c] = gld<uint2>(b + 16 + 32 * c + 8 * oct);
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int i = 8 * (j & 3);
    const uint32_t sc = j < 4 ? (h.y >> i) & 63 : ((h.w >> i) & 15) | (((h.y >> (i + 6)) & 3) << 4);
    const uint32_t mn = j < 4 ? (h.z >> i) & 63 : ((h.w >> (i + 4)) & 15) | (((h.z >> (i + 6)) & 3) << 4);
    const float a = d * (float)sc, m = dm * (float)mn;
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; e++) w[e] = __builtin_fmaf(a, (float)((byte8(q[j >> 1], e) >> (4 * (j & 1))) & 15), -m);
    put_octet(out + (size_t)j * kDWStep, w);
  }
}

__device__ __forceinline__ void octets_q6k(uint8_t *out, const uint8_t *b, int oct) {
  const float d = gq_h2f(gld<uint16_t>(b + 208));
  uint2 ql[4], qh[2];
#pragma unroll
  for (int n = 0; n < 4; n++) ql[n] = ld8(b + 32 * n + 8 * oct);
#pragma unroll
  for (int n = 0; n < 2; n++) qh[n] = ld8(b + 128 + 32 * n + 8 * oct);
#pragma unroll
  for (int st = 0; st < 8; st++) {
    const int n = st >> 2, g = st & 3;
    const float a = d * (float)(int8_t)(gld<uint16_t>(b + 192 + 8 * n + 2 * g) >> (8 * (oct >> 1)));
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t lo = (byte8(ql[2 * n + (g & 1)], e) >> (4 * (g >> 1))) & 15, hi = (byte8(qh[n], e) >> (2 * g)) & 3;
      w[e] = a * (float)((int)(lo | (hi << 4)) - 32);
    }
    put_octet(out + (size_t)st * kDWStep, w);
  }
}

__device__ __forceinline__ void octets_q8(uint8_t *out, const uint8_t *b, int oct) {
#pragma unroll
  for (int st = 0; st < 8; st++) {
    const float d = gq_h2f(gld<uint16_t>(b + 34 * st));
    const uint2 q = ld8(b + 34 * st + 2 + 8 * oct);
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; e++) w[e] = d * (float)(int8_t)byte8(q, e);
    put_octet(out + (size_t)st * kDWStep, w);
  }
}

/* One workgroup per 64 rows of a 256-row tile and 256 columns, four lanes a
 * row.  Tile row r is row 256 tile + r of w0, or with w1 (gate and up) 32-row
 * blocks of both in turn: row 128 tile + 32 (r / 64) + r % 32 of w0 where (r /
 * 32) is even, of w1 where it is odd.  Rows past `rows` are zero.
 *
 * The prompt that makes the copies waits for this; what bounds it is the 2
 * bytes a weight it writes.  us at the 8B shape, with a load a byte and a
 * workgroup per 256 rows / as it is: q and o 16.2 / 8.3, k and v 14.8 / 4.1, gate
 * + up 106 / 61 (3.9 TB/s written), down 51 / 23 (Q6_K 69 / 26); the whole
 * model 8.1 / 3.9 ms. */
template <int DT>
__global__ __launch_bounds__(256) void dense_tile_kernel(uint8_t *dst, const uint8_t *w0, const uint8_t *w1, int rows,
                                                         int K) {
  const int tile = blockIdx.x, kb = blockIdx.y, tid = threadIdx.x;
  const int r = 64 * blockIdx.z + (tid >> 2), oct = (tid & 3) ^ ((r >> 1) & 3);
  const bool up = w1 && ((r >> 5) & 1);
  const int row = w1 ? tile * 128 + 32 * (r >> 6) + (r & 31) : tile * kDN + r;
  uint8_t *out = dst + ((size_t)tile * (K / kDK) + 8 * kb) * kDWStep + 64 * r + 16 * (tid & 3);
  if (row >= rows) {
    for (int st = 0; st < 8; st++) gst<uint4>(out + (size_t)st * kDWStep, make_uint4(0, 0, 0, 0));
    return;
  }
  constexpr size_t kBlock = DT == GQ_Q4_K ? 144 : DT == GQ_Q6_K ? 210 : 8 * 34;
  const uint8_t *b = (up ? w1 : w0) + ((size_t)row * (K / 256) + kb) * kBlock;
  if constexpr (DT == GQ_Q4_K) octets_q4k(out, b, oct);
  else if constexpr (DT == GQ_Q6_K) octets_q6k(out, b, oct);
  else octets_q8(out, b, oct);
}

/* ---- the GEMM ---------------------------------------------------------- */
__device__ __forceinline__ void dma16s(const void *base, uint32_t off, uint32_t lds_addr) {
  asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(lds_addr));
}

/* A workgroup of four waves takes 64 TM tokens x 256 rows; wave (wm, wn) 32
 * TM tokens x 128 rows as TM x 4 tiles of v_mfma_f32_32x32x16_bf16.  K
 * advances 32 columns a step through an LDS ring filled by global -> LDS DMA,
 * kSlots - 1 steps ahead.  TM = 4: 16 MFMAs per 8 operand reads (1 KB each),
 * 75% of the LDS rate at the full MFMA rate; one wave per SIMD, so each half
 * step's operands are read while the other half's 16 MFMAs run, and the
 * barrier stands between the two. */
template <int TM>
struct Dense {
  static constexpr int kMT = 64 * TM;
  static constexpr int kX = kMT * kDK * 2; /* bytes of X per step */
  static constexpr int kStage = kX + kDWStep;
  static constexpr int kSlots = TM == 4 ? 5 : 6;
  static constexpr int kLds = kSlots * kStage;
  static constexpr int kDma = TM + 4; /* DMA instructions per wave and step */
  static_assert(kLds <= 160 * 1024 && (kSlots - 2) * kDma < 64, "ring");
};

template <int MODE, int TM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void dense_kernel(DnArgs a) {
  typedef Dense<TM> D;
  constexpr int NS = D::kSlots;
  extern __shared__ __attribute__((aligned(16))) uint8_t dn_smem[];
  GQ_LDS uint8_t *smem = (GQ_LDS uint8_t *)dn_smem;
  const uint32_t sbase = (uint32_t)(uintptr_t)smem;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wv >> 1, wn = wv & 1;
  const int tile = blockIdx.x, t0 = blockIdx.y * D::kMT;
  /* this part's steps s0 .. s0 + ns - 1 */
  const int nk = a.K / kDK, s0 = (int)((long)nk * blockIdx.z / a.kparts);
  const int ns = (int)((long)nk * (blockIdx.z + 1) / a.kparts) - s0;
  /* DMA: X instruction q covers 16 tokens' 64-byte slices, lane position l %
   * 4 of token l / 4 fetching the octet that the swizzle puts there.  Per-lane
   * 32-bit offsets from bases that advance in scalar registers. */
  uint32_t xoff[TM];
#pragma unroll
  for (int j = 0; j < TM; j++) {
    const int row = 16 * (TM * wv + j) + (lane >> 2), oct = (lane & 3) ^ ((row >> 1) & 3);
    xoff[j] = (uint32_t)min(t0 + row, a.T - 1) * (uint32_t)(2 * a.K) + 16u * (uint32_t)oct;
  }
  const uint8_t *xs = (const uint8_t *)a.x + (size_t)s0 * (2 * kDK);
  const uint8_t *ws = a.w + ((size_t)tile * nk + s0) * kDWStep + 4096 * wv;
  const uint32_t wlane = 16u * (uint32_t)lane;
  uint32_t dslot = sbase; /* where the next step issued goes */
  auto dma = [&](int j) { /* instruction j of the step at xs, ws */
    if (j < TM) dma16s(xs, xoff[j < TM ? j : 0], dslot + 1024u * (uint32_t)(TM * wv + j));
    else dma16s(ws + 1024 * (j - TM), wlane, dslot + D::kX + 4096u * (uint32_t)wv + 1024u * (uint32_t)(j - TM));
  };
  auto next = [&](uint32_t slot, uint32_t first) { return slot == first + (NS - 1) * D::kStage ? first : slot + D::kStage; };
  auto issued = [&]() { xs += 2 * kDK, ws += kDWStep, dslot = next(dslot, sbase); };
  for (int st = 0; st < NS - 1 && st < ns; st++) {
#pragma unroll
    for (int j = 0; j < D::kDma; j++) dma(j);
    issued();
  }
  gq_f32x16 acc[TM][4];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = gq_f32x16{};
  /* operand addresses in a slot, first half step; the second is 32 away */
  const uint32_t sw = (uint32_t)((h ^ ((r >> 1) & 3)) << 4);
  const uint32_t aoff = (uint32_t)((wm * 32 * TM + r) * 64) + sw, boff = (uint32_t)(D::kX + (wn * 128 + r) * 64) + sw;
  gq_bf16x8 fa[2][TM], fb[2][4];
  auto read = [&](uint32_t slot, int half) {
    const uint32_t x = half ? 32u : 0u;
#pragma unroll
    for (int i = 0; i < TM; i++) fa[half][i] = lld<gq_bf16x8>(smem, slot + (aoff ^ x) + 2048u * i);
#pragma unroll
    for (int j = 0; j < 4; j++) fb[half][j] = lld<gq_bf16x8>(smem, slot + (boff ^ x) + 2048u * j);
  };
  auto mma = [&](int half, int i, int j) {
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[half][i], fb[half][j], acc[i][j], 0, 0, 0);
  };
  wait_groups<D::kDma, NS - 2>(ns - 1);
  __syncthreads();
  uint32_t rslot = 0; /* step s's slot */
  read(rslot, 0);
  for (int s = 0; s < ns; s++) {
    read(rslot, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4 * TM; u++) mma(0, u >> 2, u & 3);
    __builtin_amdgcn_sched_barrier(0);
    /* this wave's copies of step s + 1 have landed once only later steps'
     * are in flight; the barrier extends that to every wave's copies, and
     * frees the slot of step s - 1 for step s + NS - 1, whose copies are
     * issued one by one between the MFMAs (a burst of them holds up the
     * wave until the memory pipeline has room) */
    if (s + 1 < ns) wait_groups<D::kDma, NS - 3>(ns - 2 - s);
    __syncthreads();
    rslot = next(rslot, 0);
    if (s + 1 < ns) read(rslot, 0);
    const bool more = s + NS - 1 < ns;
#pragma unroll
    for (int u = 0; u < D::kDma; u++) {
      __builtin_amdgcn_sched_barrier(0);
      if (more) dma(u);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = u * 4 * TM / D::kDma; q < (u + 1) * 4 * TM / D::kDma; q++) mma(1, q >> 2, q & 3);
    }
    if (more) issued();
  }
  /* token 32 i + 8 (e / 4) + 4 h + e % 4 of the wave's, row 32 j + lane % 32 */
  const int tw = t0 + wm * 32 * TM + 4 * h;
  if (MODE == MV_SWIGLU) { /* tiles 0, 2 gate and 1, 3 up of the same rows */
#pragma unroll
    for (int jj = 0; jj < 2; jj++) {
      const int n = tile * 128 + wn * 64 + 32 * jj + r;
      if (n >= a.rows[0]) continue;
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int t = tw + 32 * i + 8 * (e >> 2) + (e & 3);
          const __bf16 v = (__bf16)gq_silu_mul(acc[i][2 * jj][e], acc[i][2 * jj + 1][e]);
          if (t < a.T) gst<unsigned short>(a.act + (size_t)t * a.rows[0] + n, __builtin_bit_cast(unsigned short, v));
        }
    }
    return;
  }
  int sg = 0, tb = tile, roff = 0; /* this tile's segment, its first row among all segments' */
  while (sg + 1 < a.nseg && tb >= (a.rows[sg] + kDN - 1) / kDN) tb -= (a.rows[sg] + kDN - 1) / kDN, roff += a.rows[sg], sg++;
  const int rows = sg == 0 ? a.rows[0] : sg == 1 ? a.rows[1] : a.rows[2];
  float *yb = sg == 0 ? a.y[0] : sg == 1 ? a.y[1] : a.y[2];
  int ld = rows;
  if (a.to_parts) yb = a.part + (size_t)blockIdx.z * a.T * a.rows_total + roff, ld = a.rows_total;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int n = tb * kDN + wn * 128 + 32 * j + r;
    if (n >= rows) continue;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int t = tw + 32 * i + 8 * (e >> 2) + (e & 3);
        if (t >= a.T) continue;
        gst<float>(yb + (size_t)t * ld + n, acc[i][j][e]);
      }
  }
}

template <int MODE, int TM>
int launch_dense(const DnArgs &a, int tiles, hipStream_t s) {
  static bool attr_done = false;
  if (!attr_done) {
    (void)hipFuncSetAttribute((const void *)dense_kernel<MODE, TM>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr_done = true;
  }
  hipLaunchKernelGGL((dense_kernel<MODE, TM>), dim3(tiles, (a.T + 64 * TM - 1) / (64 * TM), a.kparts), dim3(256),
                     Dense<TM>::kLds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}

} // namespace

size_t gq_dense_bytes(int rows, int K, bool swiglu) {
  const int per = swiglu ? kDN / 2 : kDN;
  return (size_t)((rows + per - 1) / per) * (K / kDK) * kDWStep;
}

int gq_launch_dense_tile(void *dst, int dtype, const void *w0, const void *w1, int rows, int K, hipStream_t s) {
  if (rows <= 0 || K <= 0 || K % 256 || (((uintptr_t)w0 | (uintptr_t)w1) & 15)) return -1;
  const dim3 grid((rows + (w1 ? kDN / 2 : kDN) - 1) / (w1 ? kDN / 2 : kDN), K / 256, kDN / 64);
  const uint8_t *a = (const uint8_t *)w0, *b = (const uint8_t *)w1;
  if (dtype == GQ_Q4_K) hipLaunchKernelGGL(dense_tile_kernel<GQ_Q4_K>, grid, dim3(256), 0, s, (uint8_t *)dst, a, b, rows, K);
  else if (dtype == GQ_Q6_K) hipLaunchKernelGGL(dense_tile_kernel<GQ_Q6_K>, grid, dim3(256), 0, s, (uint8_t *)dst, a, b, rows, K);
  else if (dtype == GQ_Q8_0) hipLaunchKernelGGL(dense_tile_kernel<GQ_Q8_0>, grid, dim3(256), 0, s, (uint8_t *)dst, a, b, rows, K);
  else return -1;
  return hipGetLastError() == hipSuccess ? 0 : -4;
}

/* Tile height and K parts by the time they should take: rounds of
 * workgroups over the CUs, at a step's measured time each and a round's
 * start and end, and the parts written and read back.  Measured (us, tall /
 * flat tiles at their best parts): 512 tokens x 14336 gate + up rows of
 * 4096: 132 / 157; 4096 rows of 14336: 101 / 75; 1536 tokens: 360 / 417, 197
 * / 209.  rows: the launch's weight rows, in so many 256-row tiles; part_cap
 * 0: no workspace for parts. */
DnShape gq_dense_shape(int mode, int tiles, size_t rows, int T, int K, size_t part_cap, int n_cu) {
  DnShape f{4, 1};
  double best = 1e30;
  for (int tm = 4; tm >= 2; tm -= 2)
    for (int kp = 1; kp <= (mode == MV_SWIGLU || !part_cap ? 1 : kPgKParts); kp *= 2) {
      if (kp > 1 && kp * T * rows > part_cap) continue;
      const int wgs = tiles * ((T + 64 * tm - 1) / (64 * tm)) * kp;
      const int rounds = (wgs + n_cu - 1) / n_cu;
      const double us = rounds * ((double)(K / kDK) / kp * (tm == 4 ? 0.92 : 0.64) + 8.0) +
                        (kp > 1 ? 8.0 * kp * T * (double)rows / 4.0e6 : 0.0);
      if (us < best) best = us, f = DnShape{tm, kp};
    }
  return f;
}

int gq_launch_dense(int mode, const DnArgs &a0, int n_cu, hipStream_t s) {
  DnArgs a = a0;
  if (!a.x || !a.w || a.T <= 0 || a.K <= 0 || a.K % 256 || a.nseg < 1 || a.nseg > 3) return -1;
  int tiles = 0;
  a.rows_total = 0;
  for (int i = 0; i < a.nseg; i++) {
    if (a.rows[i] <= 0 || (mode != MV_SWIGLU && !a.y[i])) return -1;
    const int per = mode == MV_SWIGLU ? kDN / 2 : kDN;
    tiles += (a.rows[i] + per - 1) / per;
    a.rows_total += a.rows[i];
  }
  if (mode == MV_SWIGLU && (a.nseg != 1 || !a.act)) return -1;
  const DnShape f = gq_dense_shape(mode, tiles, a.rows_total, a.T, a.K, a.part ? a.part_cap : 0, n_cu);
  a.kparts = f.kparts;
  /* A residual launch always leaves its sums in the workspace: the RMSNorm
   * that follows adds them as it reads the row (an epilogue that reads the
   * residual back took 75 us at 512 x 4096 x 4096, one load after another). */
  a.to_parts = f.kparts > 1 || mode == MV_RESID;
  if (a.to_parts && (!a.part || (size_t)f.kparts * a.T * a.rows_total > a.part_cap)) return -1;
  if (a.kparts_out) *a.kparts_out = a.to_parts ? f.kparts : 0;
  int rc;
  if (mode == MV_SWIGLU) rc = f.tm == 4 ? launch_dense<MV_SWIGLU, 4>(a, tiles, s) : launch_dense<MV_SWIGLU, 2>(a, tiles, s);
  else rc = f.tm == 4 ? launch_dense<MV_STORE, 4>(a, tiles, s) : launch_dense<MV_STORE, 2>(a, tiles, s);
  if (rc || !a.to_parts || a.kparts_out) return rc;
  PgArgs p{};
  p.nseg = a.nseg, p.T = a.T, p.K = a.K, p.part = a.part, p.kparts = f.kparts, p.rows_total = a.rows_total;
  for (int i = 0; i < a.nseg; i++) p.seg[i].y = a.y[i], p.seg[i].rows = a.rows[i];
  return gq_launch_parts(p, mode == MV_RESID, s);
}
