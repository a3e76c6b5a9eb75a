/*
 * gq_sample.hip — sampling the next token on the device from logits already
 * there (the LM head's output), so a sampled decode step needs no logits
 * round trip (tokenizer.c:175-333 on the host copies 501 KiB per token at
 * the 8B shape).
 *
 * The reference draws one rand() per sampled token and scales it as
 * (float)rand() / (float)RAND_MAX (temperature, top-k) or in double
 * (top-p).  The caller passes that raw draw (`rnd`), so with the same libc
 * stream the device sees the same random numbers.
 *
 *   top-k (tokenizer.c:219-280): the reference keeps k slots, filled with
 *     logits 0..k-1, and for every later logit above the slots' minimum
 *     replaces that minimum (the lowest slot among equal minima).  The
 *     slots' order decides which token a given draw picks, so the kernel
 *     replays exactly that insertion sequence: logits 0..kPre-1 by one
 *     wave, 64 at a time, then every later logit above the minimum after
 *     kPre (the running minimum only rises, so nothing below it can be
 *     inserted later), gathered by all waves and inserted in index order.
 *     For k <= 64 the slots live in registers, one per lane, and a
 *     replacement's new minimum is one DPP reduction.  The softmax over the
 *     slots and the draw then run on one thread in the reference's order.
 *   top-p (tokenizer.c:282-333): stable descending sort (rocPRIM's device
 *     radix sort of (logit, index) pairs; the reference's qsort is glibc's
 *     merge sort, stable for equal logits),
 *     then the cumulative probabilities in double.
 *   temperature (tokenizer.c:187-217): the exponentials in parallel, the
 *     reference's sequential float sum and scan on one thread (see
 *     temp_kernel).
 */
#include <rocprim/device/device_radix_sort.hpp>

#include "gq_device.h"
#include "gq_internal.h"

namespace {

constexpr int kST = 1024;           /* threads of the one-workgroup kernels */
constexpr int kSW = kST / GQ_WAVE;  /* their waves */
constexpr int kPre = 4 * kST;       /* logits replayed chunk by chunk before the filter */
constexpr int kCandCap = 8192;      /* filtered candidates held in LDS */
constexpr float kRandMax = 2147483647.0f; /* RAND_MAX of glibc, as the reference casts it */

/* A float's bits mapped to an unsigned integer of the same order. */
__device__ __forceinline__ uint32_t ord_bits(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

/* 64-bit DPP move of the row operation CTRL (rows not in RM keep their own
 * value) */
template <int CTRL, int RM>
__device__ __forceinline__ uint64_t dpp64(uint64_t k) {
  const int lo = (int)(uint32_t)k, hi = (int)(uint32_t)(k >> 32);
  const uint32_t nlo = (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, CTRL, RM, 0xf, false);
  const uint32_t nhi = (uint32_t)__builtin_amdgcn_update_dpp(hi, hi, CTRL, RM, 0xf, false);
  return ((uint64_t)nhi << 32) | nlo;
}

/* The wave's smallest 64-bit key, in every lane: quad swaps, half-row and
 * row mirrors, then the row broadcasts 15 and 31 into lane 63. */
__device__ __forceinline__ uint64_t wave_min_key(uint64_t k) {
  uint64_t t;
  t = dpp64<0xb1, 0xf>(k), k = t < k ? t : k; /* quad_perm [1,0,3,2] */
  t = dpp64<0x4e, 0xf>(k), k = t < k ? t : k; /* quad_perm [2,3,0,1] */
  t = dpp64<0x141, 0xf>(k), k = t < k ? t : k; /* row_half_mirror */
  t = dpp64<0x140, 0xf>(k), k = t < k ? t : k; /* row_mirror */
  t = dpp64<0x142, 0xa>(k), k = t < k ? t : k; /* row_bcast:15 */
  t = dpp64<0x143, 0xc>(k), k = t < k ? t : k; /* row_bcast:31 */
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(k >> 32), 63);
  return ((uint64_t)hi << 32) | lo;
}

/* (value, slot) of the slots' minimum with the reference's tie rule (the
 * first slot holding the smallest value), over slots [0, k), by one wave:
 * the minimum of (value order, slot) keys */
__device__ void wave_min(const float *tv, int k, int lane, float &mv, int &mj) {
  uint64_t key = ~0ull;
  for (int s = lane; s < k; s += GQ_WAVE) {
    const float t = tv[s];
    const uint64_t c = ((uint64_t)ord_bits(t == 0.f ? 0.f : t) << 32) | (uint32_t)s; /* -0 equals +0 */
    key = c < key ? c : key;
  }
  key = wave_min_key(key);
  mj = (int)(uint32_t)key;
  mv = tv[mj];
}

/* inverse of ord_bits */
__device__ __forceinline__ float from_ord(uint32_t o) {
  return __builtin_bit_cast(float, (o & 0x80000000u) ? (o ^ 0x80000000u) : ~o);
}

/* The k slots of the reference's top-k, held by wave 0.  k <= 64: one slot
 * per lane in registers; larger k: in LDS. */
struct RegSlots {
  float v;
  int i, k, lane;
  __device__ void init(const float *x, int k_, int lane_) {
    k = k_, lane = lane_;
    v = lane < k ? x[lane] : 0.f;
    i = lane;
  }
  /* the minimum with the reference's tie rule (first slot of the smallest) */
  __device__ void minimum(float &mv, int &mj) const {
    const uint64_t key = lane < k ? ((uint64_t)ord_bits(v == 0.f ? 0.f : v) << 32) | (uint32_t)lane : ~0ull;
    const uint64_t m = wave_min_key(key);
    mj = (int)(uint32_t)m;
    mv = from_ord((uint32_t)(m >> 32));
  }
  __device__ void replace(int mj, float nv, int ni) {
    if (lane == mj) v = nv, i = ni;
  }
  __device__ void store(float *tv, int *ti) const {
    if (lane < k) tv[lane] = v, ti[lane] = i;
  }
};

struct LdsSlots {
  float *tv;
  int *ti;
  int k, lane;
  __device__ void init(const float *x, int k_, int lane_) {
    k = k_, lane = lane_;
    for (int j = lane; j < k; j += GQ_WAVE) tv[j] = x[j], ti[j] = j;
    __builtin_amdgcn_s_waitcnt(0xc07f); /* lgkmcnt(0) */
    __builtin_amdgcn_wave_barrier();
  }
  __device__ void minimum(float &mv, int &mj) const { wave_min(tv, k, lane, mv, mj); }
  __device__ void replace(int mj, float nv, int ni) {
    if (lane == 0) tv[mj] = nv, ti[mj] = ni;
    __builtin_amdgcn_s_waitcnt(0xc07f); /* the slot write lands before the rescan */
    __builtin_amdgcn_wave_barrier();
  }
  __device__ void store(float *, int *) const {}
};

/* Wave 0 replays the reference's slot updates for a group of up to 64
 * candidates held one per lane in index order (valid lanes flagged). */
template <class S>
__device__ __forceinline__ void insert_lanes(S &sl, bool valid, float v, int id, float &mv, int &mj) {
  const int lane = sl.lane;
  uint64_t live = __ballot(valid && v > mv);
  while (live) {
    const int l = __builtin_ctzll(live); /* the next candidate in index order */
    const float vl = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
    const int il = __builtin_amdgcn_readlane(id, l);
    sl.replace(mj, vl, il);
    sl.minimum(mv, mj);
    live = __ballot(valid && lane > l && v > mv);
  }
}

/* Wave 0 over logits [lo, hi) in index order, 64 at a time (the next 64
 * already loading) */
template <class S>
__device__ void scan_range(S &sl, const float *x, int lo, int hi, float &mv, int &mj) {
  const int lane = sl.lane;
  float nx = lo + lane < hi ? x[lo + lane] : 0.f;
  for (int b = lo; b < hi; b += GQ_WAVE) {
    const float v = nx;
    nx = b + GQ_WAVE + lane < hi ? x[b + GQ_WAVE + lane] : 0.f;
    insert_lanes(sl, b + lane < hi, v, b + lane, mv, mj);
  }
}

struct TopkShared {
  float tv[kMaxTopK], pr[kMaxTopK];
  int ti[kMaxTopK];
  int ci[kCandCap];
  float cv[kCandCap]; /* topk_fast_slots reads it 16 bytes at a time */
  __attribute__((aligned(16))) int wn[kSW];
  int wovf[kSW];
  float s_mv;
  int s_mj;
};

template <class S>
__device__ void topk_body(S &sl, const float *x, int V, int k, float T, int rnd, int *out, TopkShared &sh) {
  float *tv = sh.tv, *pr = sh.pr, *cv = sh.cv;
  int *ti = sh.ti, *ci = sh.ci, *wn = sh.wn, *wovf = sh.wovf;
  float &s_mv = sh.s_mv;
  int &s_mj = sh.s_mj;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  /* logits 0 .. pre-1 by wave 0 alone: the slots' first k, then in order */
  const int pre = min(V, max(kPre, k));
  if (wave == 0) {
    float mv;
    int mj;
    sl.init(x, k, lane);
    sl.minimum(mv, mj);
    scan_range(sl, x, k, pre, mv, mj);
    if (lane == 0) s_mv = mv, s_mj = mj;
  }
  __syncthreads();
  /* the rest: each wave gathers, in index order, the logits of its own
   * contiguous slice above the minimum after `pre` logits (the minimum only
   * rises, so no other logit can enter a slot later); a wave whose list
   * fills up records where it stopped */
  const float thr = s_mv;
  constexpr int kCapW = kCandCap / kSW;
  const int per = (V - pre + kSW - 1) / kSW, lo = min(V, pre + wave * per), hi = min(V, lo + per);
  int n = 0, ovf = hi;
  for (int b0 = lo; b0 < hi && ovf == hi; b0 += 8 * GQ_WAVE) {
    float vv[8]; /* eight groups' loads in flight at once */
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = b0 + u * GQ_WAVE + lane;
      vv[u] = i < hi ? x[i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int b = b0 + u * GQ_WAVE, i = b + lane;
      const bool c = i < hi && vv[u] > thr;
      const uint64_t bal = __ballot(c);
      const int cnt = __popcll(bal);
      if (ovf == hi && b < hi) {
        if (n + cnt > kCapW) {
          ovf = b;
        } else {
          const int at = n + __popcll(bal & ((1ull << lane) - 1ull));
          if (c) ci[wave * kCapW + at] = i, cv[wave * kCapW + at] = vv[u];
          n += cnt;
        }
      }
    }
  }
  if (lane == 0) wn[wave] = n, wovf[wave] = ovf;
  __syncthreads();
  /* wave 0: the gathered lists in order up to the first slice that filled
   * up, then logit by logit from there */
  if (wave == 0) {
    float mv = s_mv;
    int mj = s_mj;
    int resume = V;
    for (int w = 0; w < kSW; w++) {
      for (int q0 = 0; q0 < wn[w]; q0 += GQ_WAVE) {
        const int q = q0 + lane;
        const bool ok = q < wn[w];
        insert_lanes(sl, ok, ok ? cv[w * kCapW + q] : 0.f, ok ? ci[w * kCapW + q] : 0, mv, mj);
      }
      const int whi = min(V, min(V, pre + w * per) + per);
      if (wovf[w] < whi) {
        resume = wovf[w];
        break;
      }
    }
    if (resume < V) scan_range(sl, x, resume, V, mv, mj);
    sl.store(tv, ti);
  }
  __syncthreads();
  /* temperature softmax over the slots and the draw, in the reference's
   * order (tokenizer.c:254-276) */
  if (tid == 0) {
    float mx = tv[0];
    for (int j = 1; j < k; j++)
      if (tv[j] > mx) mx = tv[j];
    float sum = 0.f;
    for (int j = 0; j < k; j++) {
      const float p = expf((tv[j] - mx) / T);
      pr[j] = p;
      sum += p;
    }
    const float r = ((float)rnd / kRandMax) * sum;
    float acc = 0.f;
    int pick = k - 1;
    for (int j = 0; j < k; j++) {
      acc += pr[j];
      if (r <= acc) {
        pick = j;
        break;
      }
    }
    *out = ti[pick];
  }
}

/* ---- top-k over the whole chip -------------------------------------------
 * The replay above is a serial chain of insertions on one wave (about
 * k ln(V / k) of them) behind a scan of the vocabulary by one workgroup:
 * 129 us at V 128256, k 40.  The three launches below pick the same token
 * from the structure of that process:
 *   - logit i is inserted iff fewer than k of the logits before it are >= it;
 *   - every insertion evicts the smallest of the slots, so the m-th insertion
 *     evicts the m-th smallest of all the inserted logits (the first k
 *     count as inserted), and an inserted logit takes its victim's slot.
 * So once the inserted logits are known in index order, ranking them gives
 * every victim, and each survivor's slot is the end of its chain of victims.
 * Many equal logits, NaN, and inputs with more than kFastCand candidates
 * (ascending logits) go back to the replay, in the same launch.
 *   topk_top_kernel   a workgroup per slice of 1024 logits: a list of the
 *                     slice's k largest, and a few more
 *   topk_cand_kernel  a workgroup per slice: a lower bound of the k-th largest
 *                     logit before the slice, from those lists, and the
 *                     slice's logits that may exceed it, in index order
 *   topk_pick_kernel  one workgroup: the inserted logits, their ranks and
 *                     slots, then the softmax and the draw as the replay has
 *                     them
 * Bounded by the latency of the dependent launches and of the last one's
 * steps, not by the 0.5 MB of logits: V 128256, k 40: 4.4 + 8.5 + 20 us
 * against the replay's 105 us; a whole gq_hip_sample_dev call 125 -> 41 us
 * (k 200: 717 -> 159, k 1: 55 -> 28; V 1024, k 1: 27 -> 24).  Kernels this
 * short are also bound by fetching their code: bisections unrolled over
 * registers in place of the histograms ran 10 + 10 us for the first two
 * launches. */
constexpr int kSlice = 1024;      /* logits per slice */
constexpr int kFastK = 256;       /* largest k: the first slice's groups and the lists are sized for it */
constexpr int kFastSlices = 256;  /* vocabularies up to 262144 */
constexpr int kFastCand = 4096;   /* candidates the last launch holds (ranked pairwise) */
constexpr int kListPer = 10;      /* list entries per thread in topk_cand_kernel */
constexpr int kBins = 256;

/* what the three launches hand on, in the context's workspace */
struct TopkWs {
  float *list; /* [slices][ls] of each slice's largest, -inf where it has fewer */
  float *low;  /* [slices] the slice has k logits that reach this (-inf: fewer) */
  int *nan;    /* [slices] the slice holds a NaN */
  int *cnt;    /* [slices] candidates */
  float *cv;   /* [slices][kSlice] their logits */
  int *ci;     /* [slices][kSlice] their indices */
};

/* list entries a slice: k and room for what shares the k-th largest's bin */
__host__ __device__ constexpr int list_stride(int k) { return k + (k + 1) / 2; }

__device__ __forceinline__ uint32_t topk_key(float v) { return ord_bits(v == 0.f ? 0.f : v); /* -0 equals +0 */ }

/* sum of NW counts (16-byte aligned, NW % 4 == 0) */
template <int NW>
__device__ __forceinline__ int block_total(const int *sc) {
  int t = 0;
#pragma unroll
  for (int g = 0; g < NW; g += 4) {
    const int4 u = *(const int4 *)(sc + g);
    t += (u.x + u.y) + (u.z + u.w);
  }
  return t;
}

/* The k-th largest is bounded from below with a histogram of the value: bin
 * 0 below lo, then kBins - 1 equal steps.  bin() never decreases with v, so
 * the logits of bins >= b are the largest ones, and where they are at least
 * k the k-th largest is one of them.  Logits above hi fall into the last
 * bin; an infinite or empty range puts all from lo on into bin 1. */
struct TopkBins {
  float lo, scale;
  __device__ TopkBins(float lo_, float hi) : lo(lo_), scale(hi > lo_ ? (float)(kBins - 1) / (hi - lo_) : 0.f) {}
  __device__ int bin(float v) const { return v < lo ? 0 : 1 + (int)fminf(fmaxf((v - lo) * scale, 0.f), (float)(kBins - 2)); }
};

/* The largest bin b whose logits and those above it are at least k (0 when
 * all are fewer), by one wave. */
__device__ __forceinline__ int topk_bin(const int *hist, int k) {
  const int lane = threadIdx.x & 63;
  const int4 h = *(const int4 *)(hist + 4 * (GQ_WAVE - 1 - lane)); /* lane 0: the top four bins */
  const int t = (h.x + h.y) + (h.z + h.w);
  int inc = t;
#pragma unroll 1
  for (int o = 1; o < GQ_WAVE; o <<= 1) {
    const int u = __shfl_up(inc, o);
    if (lane >= o) inc += u;
  }
  const uint64_t bal = __ballot(inc >= k);
  if (!bal) return 0;
  const int l = __builtin_ctzll(bal);
  const int above = inc - t, b0 = 4 * (GQ_WAVE - 1 - lane); /* counted above this lane's bins */
  const int b = above + h.w >= k ? b0 + 3 : above + h.w + h.z >= k ? b0 + 2 : above + h.w + h.z + h.y >= k ? b0 + 1 : b0;
  return __builtin_amdgcn_readlane(b, l);
}

__device__ __forceinline__ float finite_low(float v) { return v == -INFINITY ? INFINITY : v; } /* for a minimum */

__global__ __launch_bounds__(256) void topk_top_kernel(const float *x, int V, int k, TopkWs w) {
  constexpr int NR = kSlice / 256, NW = 4;
  __shared__ __attribute__((aligned(16))) int hist[kBins], sc[NW];
  __shared__ float smx[NW], smn[NW], slow[NW];
  __shared__ int snan[NW], s_bin;
  const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, base = s * kSlice;
  float v[NR], mx = -INFINITY, mn = INFINITY;
  bool nan = false;
  hist[tid] = 0;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    v[r] = x[min(base + r * 256 + tid, V - 1)];
    nan |= v[r] != v[r];
    mx = fmaxf(mx, v[r]), mn = fminf(mn, finite_low(v[r]));
  }
  mx = gq_wave_max(mx), mn = -gq_wave_max(-mn);
  const bool any = __ballot(nan) != 0;
  if (lane == 0) smx[wave] = mx, smn[wave] = mn, snan[wave] = any;
  __syncthreads();
  const TopkBins B(fminf(fminf(smn[0], smn[1]), fminf(smn[2], smn[3])), fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3])));
#pragma unroll
  for (int r = 0; r < NR; r++)
    if (base + r * 256 + tid < V) atomicAdd(&hist[B.bin(v[r])], 1);
  __syncthreads();
  if (wave == 0) {
    const int b = topk_bin(hist, k);
    if (lane == 0) s_bin = b;
  }
  __syncthreads();
  /* the list: these bins' logits, the first list_stride(k) in any order */
  const int bin = s_bin, ls = list_stride(k);
  float low = INFINITY;
  int n = 0;
  uint64_t bal[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const bool c = base + r * 256 + tid < V && B.bin(v[r]) >= bin;
    if (c) low = fminf(low, v[r]);
    bal[r] = __ballot(c);
    n += __popcll(bal[r]);
  }
  low = -gq_wave_max(-low);
  if (lane == 0) sc[wave] = n, slow[wave] = low;
  __syncthreads();
  int at = 0;
  for (int g = 0; g < wave; g++) at += sc[g];
  const int total = block_total<NW>(sc);
  float *list = w.list + (size_t)s * ls;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int j = at + __popcll(bal[r] & ((1ull << lane) - 1ull));
    if (((bal[r] >> lane) & 1) && j < ls) list[j] = v[r];
    at += __popcll(bal[r]);
  }
  for (int j = total + tid; j < ls; j += 256) list[j] = -INFINITY;
  if (tid == 0) {
    w.low[s] = total < k ? -INFINITY : fminf(fminf(slow[0], slow[1]), fminf(slow[2], slow[3]));
    w.nan[s] = (snan[0] | snan[1]) | (snan[2] | snan[3]);
  }
}

/* Slice s > 0: its logits that may exceed the k-th largest of the lists of
 * the slices before it (of the first of them where all lists together are
 * longer than kListPer a thread).  Slice 0: its first p0 logits (p0 a power
 * of two >= k), then group g, the logits [p0 2^g, p0 2^(g+1)), against the
 * first p0 2^g.  In index order. */
__global__ __launch_bounds__(kSlice) void topk_cand_kernel(const float *x, int V, int k, TopkWs w) {
  constexpr int NW = kSlice / GQ_WAVE, NG = 4;
  __shared__ __attribute__((aligned(16))) int hist[NG * kBins], sc[NW];
  __shared__ float smx[NW], smn[NW];
  __shared__ int s_bin[NG];
  const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = s * kSlice + tid;
  const float own = i < V ? x[i] : -INFINITY;
  static_assert(NG * kBins == kSlice, "one bin a thread");
  hist[tid] = 0;
  const int ls = list_stride(k);
  const int P = min(s, kSlice * kListPer / ls); /* lists used */
  int lp0 = 6;
  while ((1 << lp0) < k) lp0++;
  float key[kListPer], mx = -INFINITY, mn = INFINITY;
#pragma unroll
  for (int r = 0; r < kListPer; r++) {
    const int j = r * kSlice + tid;
    key[r] = s > 0 ? (j < P * ls ? w.list[j] : -INFINITY) : (r == 0 ? own : -INFINITY);
    mx = fmaxf(mx, key[r]);
  }
  /* the bins' range: slice 0 its own; the others from the largest value that
   * k logits of one of the lists reach */
  if (s == 0) mn = finite_low(own);
  else
    for (int j = lane; j < P; j += GQ_WAVE) mn = fminf(mn, -w.low[j]); /* -max */
  mx = gq_wave_max(mx), mn = -gq_wave_max(-mn);
  if (lane == 0) smx[wave] = mx, smn[wave] = mn;
  __syncthreads();
  for (int g = 0; g < NW; g++) mx = fmaxf(mx, smx[g]), mn = fminf(mn, smn[g]);
  const TopkBins B(s == 0 ? mn : -mn, mx);
  if (s > 0) {
#pragma unroll
    for (int r = 0; r < kListPer; r++)
      if (r * kSlice + tid < P * ls) atomicAdd(&hist[B.bin(key[r])], 1);
  } else if (i < V) {
    for (int g = 0; g < NG; g++)
      if (tid < (1 << (lp0 + g))) atomicAdd(&hist[g * kBins + B.bin(own)], 1);
  }
  __syncthreads();
  if (wave < (s > 0 ? 1 : NG)) {
    const int b = topk_bin(hist + wave * kBins, k);
    if (lane == 0) s_bin[wave] = b;
  }
  __syncthreads();
  /* slice 0: logit tid's group */
  const int g = s > 0 ? 0 : 31 - __builtin_clz(max(tid, 1)) - lp0;
  const bool take = i < V && (g < 0 || B.bin(own) >= s_bin[min(max(g, 0), NG - 1)]);
  const uint64_t bal = __ballot(take);
  if (lane == 0) sc[wave] = __popcll(bal);
  __syncthreads();
  int at = __popcll(bal & ((1ull << lane) - 1ull));
  for (int q = 0; q < wave; q++) at += sc[q];
  if (take) {
    const size_t j = (size_t)s * kSlice + at;
    w.cv[j] = own, w.ci[j] = i;
  }
  if (tid == 0) w.cnt[s] = block_total<NW>(sc);
}

/* sum over aligned groups of eight lanes */
__device__ __forceinline__ int oct_sum(int v) {
  v += __shfl_xor(v, 1, GQ_WAVE);
  v += __shfl_xor(v, 2, GQ_WAVE);
  return v + __shfl_xor(v, 4, GQ_WAVE);
}

constexpr int kTies = kSW; /* groups of equal logits, and members of one, that are sorted one by one */

/* the slot of the p-th inserted logit: its victim's, and so on down to one
 * of the first k (a victim was inserted earlier, so the chain ends) */
__device__ __forceinline__ int slot_of(const int *by, int k, int p) {
  while (p >= k) {
    const int f = by[p - k];
    if (f >= p) return p;
    p = f;
  }
  return p;
}

/* The candidates' inserted logits, their slots (tv, ti in `sh`); false when
 * the replay has to decide (uniform over the workgroup). */
__device__ bool topk_fast_slots(int slices, int k, const TopkWs &w, TopkShared &sh) {
  static_assert(2 * kFastCand <= kCandCap, "the candidates and the inserted fit the replay's lists");
  uint32_t *key = (uint32_t *)sh.cv, *ikey = key + kFastCand;
  int *idx = sh.ci, *iidx = idx + kFastCand;
  int *offs = (int *)sh.pr; /* kFastSlices + 1 */
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  static_assert(kMaxTopK > kFastSlices, "offsets fit pr");
  if (wave == 0) { /* exclusive scan of the counts, four slices a lane */
    int c[4], t = 0, bad = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int s = 4 * lane + q;
      c[q] = s < slices ? w.cnt[s] : 0;
      bad |= s < slices ? w.nan[s] : 0;
      t += c[q];
    }
    int inc = t;
#pragma unroll
    for (int o = 1; o < GQ_WAVE; o <<= 1) {
      const int u = __shfl_up(inc, o);
      if (lane >= o) inc += u;
    }
    int at = inc - t;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      offs[4 * lane + q] = at;
      at += c[q];
    }
    const bool any = __ballot(bad != 0) != 0;
    if (lane == GQ_WAVE - 1) offs[kFastSlices] = any ? kFastCand + 1 : at;
    if (lane == 0) sh.s_mj = 0;
  }
  __syncthreads();
  const int N = offs[kFastSlices];
  if (N > kFastCand) return false;
  for (int p = tid; p < N; p += kST) {
    int lo = 0, hi = slices - 1; /* the last slice whose offset is <= p */
    while (lo < hi) {
      const int m = (lo + hi + 1) >> 1;
      if (offs[m] <= p) lo = m;
      else hi = m - 1;
    }
    const int j = lo * kSlice + (p - offs[lo]);
    key[p] = topk_key(w.cv[j]), idx[p] = w.ci[j];
  }
  __syncthreads();
  /* inserted: fewer than k of the candidates before it are >= it.  Eight
   * lanes count for one candidate, four of the others at a time. */
  const int sub = tid & 7, grp = tid >> 3; /* 128 candidates at once */
  for (int p = grp; p < N; p += kST / 8) {
    const uint32_t a = key[p];
    int c = 0;
#pragma unroll 2
    for (int j = 4 * sub; j + 4 <= p; j += 32) {
      const uint4 u = *(const uint4 *)(key + j);
      c += (u.x >= a) + (u.y >= a) + (u.z >= a) + (u.w >= a);
    }
    if (sub < (p & 3)) c += key[(p & ~3) + sub] >= a;
    c = oct_sum(c);
    if (sub == 0) iidx[p] = c < k; /* whether p is inserted, until the lists below */
  }
  __syncthreads();
  int M = 0;
  for (int b = 0; b < N; b += kST) {
    const int p = b + tid;
    const bool ins = p < N && iidx[p] != 0;
    const uint64_t bal = __ballot(ins);
    if (lane == 0) sh.wn[wave] = __popcll(bal);
    __syncthreads();
    int at = M;
    for (int g = 0; g < wave; g++) at += sh.wn[g];
    M += block_total<kSW>(sh.wn);
    at += __popcll(bal & ((1ull << lane) - 1ull));
    if (ins) ikey[at] = key[p], iidx[at] = idx[p]; /* at <= p: flags from b + kST on are untouched */
    __syncthreads();
  }
  /* ascending ranks; rank r's element in by[].  Up to three entries past M
   * are above every logit. */
  if (tid < 3 && M + tid < kFastCand) ikey[M + tid] = ~0u;
  __syncthreads();
  int *by = (int *)key;
  for (int b = 0; b < M; b += kST / 8) {
    const int p = b + grp;
    const uint32_t a = p < M ? ikey[p] : 0u;
    int c = 0, e = 0, f = 0;
#pragma unroll 2
    for (int j = 4 * sub; j < M; j += 32) {
      const uint4 u = *(const uint4 *)(ikey + j);
      c += (u.x < a) + (u.y < a) + (u.z < a) + (u.w < a);
      e += (u.x == a) + (u.y == a) + (u.z == a) + (u.w == a);
    }
    c = oct_sum(c), e = oct_sum(e);
    if (e > 1) { /* equal ones before p */
      for (int j = sub; j < p; j += 8) f += ikey[j] == a;
      f = oct_sum(f);
    }
    if (sub == 0 && p < M) {
      by[c + f] = p;
      if (e > 1 && f == 0 && c < M - k) { /* equal logits, some of them evicted */
        const int g = atomicAdd(&sh.s_mj, 1);
        if (g < kTies) sh.wovf[g] = c << 16 | min(e, 0xffff);
      }
    }
  }
  __syncthreads();
  /* Equal logits are evicted from the lowest slot up.  All of them are in the
   * slots before the first is evicted (one equal to the minimum is not
   * inserted), and their slots depend on smaller victims only: so group by
   * group, in ascending order, sorted by slot. */
  const int ties = sh.s_mj;
  if (ties) {
    bool many = ties > kTies;
    for (int g = 0; g < min(ties, kTies); g++) many |= (sh.wovf[g] & 0xffff) > kTies;
    if (many) return false;
    __syncthreads();
    if (tid == 0) {
      sh.s_mj = 0;
      for (int n = 0; n < ties; n++) {
        int g = n;
        for (int q = n + 1; q < ties; q++) g = (sh.wovf[q] >> 16) < (sh.wovf[g] >> 16) ? q : g;
        const int w0 = sh.wovf[g];
        sh.wovf[g] = sh.wovf[n];
        const int c = w0 >> 16, e = w0 & 0xffff;
        for (int i = 1; i < e; i++) /* insertion sort */
          for (int j = i; j > 0; j--) {
            const int u = by[c + j - 1], v = by[c + j];
            if (slot_of(by, k, u) < slot_of(by, k, v)) break;
            by[c + j - 1] = v, by[c + j] = u;
          }
      }
    }
    __syncthreads();
  }
  /* element k + m took the slot of the m-th smallest; the k largest survive */
  for (int r = M - k + tid; r < M; r += kST) {
    const int p = by[r];
    const int e = slot_of(by, k, p);
    if (e < k) sh.tv[e] = from_ord(ikey[p]), sh.ti[e] = iidx[p];
    else sh.s_mj = 1;
  }
  __syncthreads();
  return sh.s_mj == 0;
}

/* The softmax over the slots and the draw of topk_body by one wave.  The
 * maximum does not depend on the order; the running float sum is the
 * reference's, each slot's lane keeping its value, and the draw's running
 * sum is that same sum. */
__device__ void topk_draw(int k, float T, int rnd, int *out, TopkShared &sh) {
  const int lane = threadIdx.x;
  if (lane >= GQ_WAVE) return;
  float mx = -INFINITY;
  for (int j = lane; j < k; j += GQ_WAVE) mx = fmaxf(mx, sh.tv[j]);
  mx = gq_wave_max(mx);
  float acc = 0.f;
  for (int b = 0; b < k; b += GQ_WAVE) {
    const int n = min(k - b, GQ_WAVE);
    const float p = lane < n ? expf((sh.tv[b + lane] - mx) / T) : 0.f;
    float mine = 0.f;
    for (int j = 0; j < n; j++) {
      acc += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), j));
      mine = lane == j ? acc : mine;
    }
    if (lane < n) sh.pr[b + lane] = mine; /* read back by the same lane */
  }
  const float r = ((float)rnd / kRandMax) * acc;
  int pick = k - 1;
  for (int b = 0; b < k; b += GQ_WAVE) {
    const uint64_t hit = __ballot(b + lane < k && r <= sh.pr[b + lane]);
    if (hit) {
      pick = b + __builtin_ctzll(hit);
      break;
    }
  }
  if (lane == 0) *out = sh.ti[pick];
}

__global__ __launch_bounds__(kST) void topk_pick_kernel(const float *x, int V, int k, float T, int rnd, int slices,
                                                        TopkWs w, int *out) {
  __shared__ __attribute__((aligned(16))) TopkShared sh;
  if (topk_fast_slots(slices, k, w, sh)) {
    topk_draw(k, T, rnd, out, sh);
    return;
  }
  __syncthreads();
  if (k <= GQ_WAVE) {
    RegSlots sl;
    topk_body(sl, x, V, k, T, rnd, out, sh);
  } else {
    LdsSlots sl;
    sl.tv = sh.tv, sl.ti = sh.ti;
    topk_body(sl, x, V, k, T, rnd, out, sh);
  }
}

size_t topk_ws_layout(int vocab, char *base, TopkWs *w) {
  const size_t S = (size_t)(vocab + kSlice - 1) / kSlice;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *p = base ? base + off : nullptr;
    off += (bytes + 255) & ~(size_t)255;
    return p;
  };
  TopkWs t;
  t.list = (float *)take(4 * S * list_stride(kFastK));
  t.low = (float *)take(4 * S);
  t.nan = (int *)take(4 * S);
  t.cnt = (int *)take(4 * S);
  t.cv = (float *)take(4 * S * kSlice);
  t.ci = (int *)take(4 * S * kSlice);
  if (w) *w = t;
  return off;
}

__global__ __launch_bounds__(kST) void topk_kernel(const float *x, int V, int k, float T, int rnd, int *out) {
  __shared__ TopkShared sh;
  if (k <= GQ_WAVE) {
    RegSlots sl;
    topk_body(sl, x, V, k, T, rnd, out, sh);
  } else {
    LdsSlots sl;
    sl.tv = sh.tv, sl.ti = sh.ti;
    topk_body(sl, x, V, k, T, rnd, out, sh);
  }
}

/* Block-wide exclusive scan of one double per thread; returns the prefix,
 * *total gets the sum (all threads). */
__device__ double block_scan(double v, double *total, double *sw) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double inc = v;
#pragma unroll
  for (int o = 1; o < GQ_WAVE; o <<= 1) {
    const double t = __shfl_up(inc, o);
    if (lane >= o) inc += t;
  }
  if (lane == GQ_WAVE - 1) sw[wave] = inc;
  __syncthreads();
  double off = 0.0, tot = 0.0;
#pragma unroll
  for (int w = 0; w < kSW; w++) {
    off += w < wave ? sw[w] : 0.0;
    tot += sw[w];
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

__device__ float block_max(float v, float *sw) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = gq_wave_max(v);
  if (lane == 0) sw[wave] = v;
  __syncthreads();
  float m = sw[0];
#pragma unroll
  for (int w = 1; w < kSW; w++) m = fmaxf(m, sw[w]);
  __syncthreads();
  return m;
}

/* The first index i in [0, n) whose inclusive running sum of w(i) reaches r
 * (n - 1 when none does); w(i) summed in double, each thread over one
 * contiguous segment. */
template <typename W>
__device__ int first_reaching(W w, int n, double r, double *sw, int *s_pick) {
  const int tid = threadIdx.x, seg = (n + kST - 1) / kST, lo = min(tid * seg, n), hi = min(lo + seg, n);
  double part = 0.0;
  for (int i = lo; i < hi; i++) part += w(i);
  double tot;
  const double before = block_scan(part, &tot, sw);
  if (tid == 0) *s_pick = n - 1;
  __syncthreads();
  if (before < r && r <= before + part) {
    /* the running sum reaches r inside this segment (its last element when
     * the sequential sum rounds just below before + part) */
    double acc = before;
    int found = hi - 1;
    for (int i = lo; i < hi; i++) {
      acc += w(i);
      if (r <= acc) {
        found = i;
        break;
      }
    }
    atomicMin(s_pick, found);
  } else if (r <= before && tid == 0) {
    atomicMin(s_pick, 0);
  }
  __syncthreads();
  return *s_pick;
}

/* softmax(x / T) over the vocabulary and one draw (tokenizer.c:187-217).
 * The reference sums the probabilities sequentially in float, and over a
 * large vocabulary that sum's rounding moves the cumulative boundaries by
 * far more than a last bit (a double sum picks a different token for about
 * one draw in four at 128256 entries), so the two sequential loops run as
 * written, on one thread: the workgroup computes the exponentials in
 * parallel and stages them through LDS in chunks of kChunkP. */
constexpr int kChunkP = 32768;

constexpr int kCkMax = 4096; /* 64-entry blocks: vocabularies up to 262144 */

__global__ __launch_bounds__(kST) void temp_kernel(const float *x, int V, float T, int rnd, float *prob, int *out) {
  __shared__ float sf[kSW];
  __shared__ float chunk[kChunkP];
  __shared__ float ck[kCkMax + 1]; /* running sum before each 64-entry block, then the total */
  __shared__ float s_r;
  __shared__ int s_blk, s_pick;
  const int tid = threadIdx.x;
  float m = -INFINITY;
  for (int i = tid; i < V; i += kST) m = fmaxf(m, x[i]);
  const float mx = block_max(m, sf);
  for (int i = tid; i < V; i += kST) prob[i] = expf((x[i] - mx) / T);
  /* the reference's running float sum, one thread, its value recorded at
   * the start of every 64-entry block */
  float sum = 0.f;
  for (int base = 0; base < V; base += kChunkP) {
    const int n = min(kChunkP, V - base);
    __syncthreads();
    for (int i = tid; i < n; i += kST) chunk[i] = prob[base + i];
    __syncthreads();
    if (tid == 0)
      for (int b = 0; b < n; b += 64) {
        ck[(base + b) >> 6] = sum;
        const int e = min(64, n - b);
        if (e == 64) {
#pragma unroll
          for (int j = 0; j < 64; j++) sum += chunk[b + j];
        } else {
          for (int j = 0; j < e; j++) sum += chunk[b + j];
        }
      }
  }
  const int nblk = (V + 63) >> 6;
  if (tid == 0) ck[nblk] = sum, s_r = ((float)rnd / kRandMax) * sum, s_blk = nblk, s_pick = V - 1;
  __syncthreads();
  /* the first block whose closing sum reaches r (sums never decrease) ... */
  const float r = s_r;
  for (int q = tid; q < nblk; q += kST)
    if (r <= ck[q + 1]) {
      atomicMin(&s_blk, q);
      break;
    }
  __syncthreads();
  /* ... then its 64 additions again, from its opening sum */
  if (tid == 0 && s_blk < nblk) {
    float acc = ck[s_blk];
    const int lo = s_blk << 6, hi = min(lo + 64, V);
    for (int i = lo; i < hi; i++) {
      acc += prob[i];
      if (r <= acc) {
        s_pick = i;
        break;
      }
    }
  }
  __syncthreads();
  if (tid == 0) *out = s_pick;
}

/* top-p over the logits sorted in descending order (keys) with their token
 * ids (ids), tokenizer.c:296-333 */
__global__ __launch_bounds__(kST) void topp_kernel(const float *keys, const int *ids, int V, float p, float T, int rnd,
                                                    int *out) {
  __shared__ double sw[kSW];
  __shared__ int s_pick;
  const float mx = keys[0];
  auto w = [&](int i) { return (double)expf((keys[i] - mx) / T); };
  double tot = 0.0;
  {
    const int seg = (V + kST - 1) / kST, lo = min((int)threadIdx.x * seg, V), hi = min(lo + seg, V);
    double part = 0.0;
    for (int i = lo; i < hi; i++) part += w(i);
    (void)block_scan(part, &tot, sw);
  }
  /* cutoff: how many leading tokens until the cumulative share reaches p */
  const double tot_c = tot;
  auto share = [&](int i) { return w(i) / tot_c; };
  const int cutoff = first_reaching(share, V, (double)p, sw, &s_pick) + 1;
  /* the draw over the first `cutoff` tokens */
  double cut = 0.0;
  {
    const int seg = (cutoff + kST - 1) / kST, lo = min((int)threadIdx.x * seg, cutoff), hi = min(lo + seg, cutoff);
    double part = 0.0;
    for (int i = lo; i < hi; i++) part += w(i);
    (void)block_scan(part, &cut, sw);
  }
  const double r = ((double)rnd / 2147483647.0) * cut;
  const int pick = first_reaching(w, cutoff, r, sw, &s_pick);
  if (threadIdx.x == 0) *out = ids[pick];
}

__global__ void iota_kernel(int *v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = i;
}

} // namespace

size_t gq_sample_ws_bytes(int vocab) {
  size_t bytes = 0;
  (void)rocprim::radix_sort_pairs_desc(nullptr, bytes, (const float *)nullptr, (float *)nullptr,
                                       (const int *)nullptr, (int *)nullptr, (size_t)vocab);
  return bytes;
}

/* The three-launch top-k takes every k and vocabulary its lists are sized
 * for.  Larger k replays: a longer list a slice leaves fewer slices to bound
 * the rest with, and the candidates no longer fit. */
size_t gq_sample_topk_bytes(int vocab, int top_k) {
  if (top_k <= 0 || top_k > kFastK || vocab > kFastSlices * kSlice) return 0;
  return topk_ws_layout(vocab, nullptr, nullptr);
}

int gq_launch_sample(const float *logits, int vocab, float temperature, int top_k, float top_p, int rnd,
                     const SampleWs &ws, int *out, hipStream_t s) {
  if (vocab <= 0 || !logits || !out) return -1;
  if (temperature <= 0.0f) return 1; /* greedy: the argmax path */
  if (top_k > 0 && top_k < vocab) {
    if (top_k > kMaxTopK) return -2;
    if (ws.topk && ws.topk_cap >= vocab && gq_sample_topk_bytes(vocab, top_k)) {
      TopkWs w;
      (void)topk_ws_layout(vocab, (char *)ws.topk, &w);
      const int slices = (vocab + kSlice - 1) / kSlice;
      hipLaunchKernelGGL(topk_top_kernel, dim3(slices), dim3(256), 0, s, logits, vocab, top_k, w);
      hipLaunchKernelGGL(topk_cand_kernel, dim3(slices), dim3(kSlice), 0, s, logits, vocab, top_k, w);
      hipLaunchKernelGGL(topk_pick_kernel, dim3(1), dim3(kST), 0, s, logits, vocab, top_k, temperature, rnd, slices, w,
                         out);
      return hipGetLastError() == hipSuccess ? 0 : -4;
    }
    hipLaunchKernelGGL(topk_kernel, dim3(1), dim3(kST), 0, s, logits, vocab, top_k, temperature, rnd, out);
  } else if (top_p < 1.0f) {
    if (top_p <= 0.0f) return 1; /* greedy (tokenizer.c:287) */
    if (!ws.keys || !ws.ids_in || !ws.ids || !ws.sort_tmp || ws.cap < vocab) return -1;
    hipLaunchKernelGGL(iota_kernel, dim3((vocab + 255) / 256), dim3(256), 0, s, ws.ids_in, vocab);
    size_t bytes = ws.sort_bytes;
    if (rocprim::radix_sort_pairs_desc(ws.sort_tmp, bytes, logits, ws.keys, ws.ids_in, ws.ids, (size_t)vocab, 0,
                                       8 * (unsigned)sizeof(float), s) != hipSuccess)
      return -4;
    hipLaunchKernelGGL(topp_kernel, dim3(1), dim3(kST), 0, s, ws.keys, ws.ids, vocab, top_p, temperature, rnd, out);
  } else {
    if (!ws.keys || ws.cap < vocab || vocab > 64 * kCkMax) return -1;
    hipLaunchKernelGGL(temp_kernel, dim3(1), dim3(kST), 0, s, logits, vocab, temperature, rnd, ws.keys, out);
  }
  return hipGetLastError() == hipSuccess ? 0 : -4;
}
