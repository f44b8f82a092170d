// Device sampler: the reference's sample_advanced (src/model.c:132-361) with
// filter_and_sample (src/model.c:67-127) and the XorShift64* generator
// (src/utils.c:117-140), bit for bit.
//
// The O(V) passes are spread over kFront blocks, each owning a contiguous
// segment of the vocabulary:
//   k_samp_scale  temperature scaling in place and the segment's max logit
//                 (or the LM head does both, with its own blocks' maxima);
//   k_samp_hist   with the global max, the 128-bucket histogram (global
//                 atomics of per-block counts) and the segment's
//                 "pre-candidates" in index order: the logits at or above the
//                 lowest threshold the extraction can use (the histogram's
//                 last bucket, or the min_p threshold), a superset of the
//                 candidates.
//   k_samp_probs  (no top-k, see tries_parallel) the probabilities, and per
//                 value bucket their count and sum.
// k_sample then runs the rest on one 1024-thread block: the cutoff bucket,
// the candidates filtered from the pre-candidate lists in order, selection,
// softmax, sorting and the draw, the step bookkeeping and the next token's
// embedding.  (Pass 2 and this in one kernel, with a block counter and
// device-scope fences handing over to the last block, measured 32 us per
// token against about 14 for the two launches.)
// With top-k, the steps whose result depends on their order stay sequential on
// one thread, in the reference's order: the heap selection (its array order
// feeds the sums), every double sum, and the CDF walk.  Without top-k the same
// sums in any order decide nearly every draw (draw_parallel); the sequential
// steps remain for the draws they leave open.  Sorting is stable
// like glibc's qsort (a merge sort for these sizes), keyed on the value.
// Float-to-int bucket indices follow x86 cvttss2si (out of range -> INT_MIN).
#include "bm_common.h"
#include "bm_exact.h"
#include "bm_dev.h"
#include "bm_libm.h"

namespace bm {

struct SampleParams {
  float temp, min_p, top_p;
  int top_k;
};

struct Cand {  // token_prob_t (src/bitmamba.h:98-102)
  int id;
  float val;
};

namespace {

constexpr int kThreads = 1024;
constexpr int kBuckets = 128;      // HIST_BUCKETS (src/model.c:131)
constexpr int kPartial = 256;      // PARTIAL_K (src/model.c:319)
constexpr int kStage = 4096;       // candidates staged in LDS per serial pass
constexpr int kCtlPos = 0, kCtlDone = 1, kCtlStep = 2, kCtlHcount = 3, kCtlToken = 4;
constexpr int kDoneArmed = 1, kDoneStopped = 2;  // the done word (bm_decode.hip)

// a decode stopped at its end token: the front kernels (given the done
// word only in a gated step graph) return at once; k_sample and
// k_sample_greedy skip their stores at the end
__device__ __forceinline__ bool step_stopped(const int* ctl) {
  return ctl && __builtin_amdgcn_readfirstlane(ctl[kCtlDone]) == kDoneStopped;
}
constexpr int kHist = 256;
constexpr int kFront = 64;          // blocks of the O(V) passes (one wave of partials)
constexpr int kFrontThreads = 256;
static_assert(kFront % (kThreads / 64) == 0, "whole pre-candidate lists per wave");
constexpr int kMaxVocab = 256000;  // MAX_VOCAB of the loader (src/bitmamba.h:55)

// vocabulary segment of each front block: a multiple of 4 entries
__host__ __device__ __forceinline__ int front_seg(int V) { return ((V + kFront - 1) / kFront + 3) & ~3; }

// Buckets of the draw without top-k: a probability's leading bits (sign,
// exponent, 4 bits of the mantissa), in value order; probabilities are <= 1
constexpr int kPShift = 19;
constexpr int kPBuckets = 2048;
static_assert((0x3f800000u >> kPShift) < kPBuckets, "1.0f has a bucket");
__device__ __forceinline__ int p_bucket(float v) {
  return min((int)(__float_as_uint(v) >> kPShift), kPBuckets - 1);
}

// scratch: probs[V], pre[kFront * seg] (also the radix sort's second
// buffer), esum[kFront], psum[kFront], bsum[kPBuckets], pv[kFront * seg]
// (beside pre: exp(logit - max), then the probability), bcnt[kPBuckets],
// pmax[kFront], pcnt[kFront], hist[kBuckets], scaled (whether k_samp_probs
// could form the probabilities).  hist is zero between calls: k_samp_scale
// clears it, and so does k_sample after use.
struct Scratch {
  Cand* probs;
  Cand* pre;
  double* esum;
  double* psum;
  double* bsum;
  float* pv;
  int* bcnt;
  float* pmax;
  int* pcnt;
  int* hist;
  int* scaled;
};
__host__ __device__ __forceinline__ Scratch scratch_of(void* base, int V) {
  Scratch s;
  // from the first 16-byte boundary, and an even number of 8-byte entries, so
  // that pv starts on 16 bytes
  s.probs = (Cand*)(((uintptr_t)base + 15) & ~(uintptr_t)15);
  s.pre = s.probs + (V + 1) / 2 * 2;
  s.esum = (double*)(s.pre + (size_t)kFront * front_seg(V));
  s.psum = s.esum + kFront;
  s.bsum = s.psum + kFront;
  s.pv = (float*)(s.bsum + kPBuckets);
  s.bcnt = (int*)(s.pv + (size_t)kFront * front_seg(V));
  s.pmax = (float*)(s.bcnt + kPBuckets);
  s.pcnt = (int*)(s.pmax + kFront);
  s.hist = s.pcnt + kFront;
  s.scaled = s.hist + kBuckets;
  return s;
}

// where the token goes: with ctl, the step bookkeeping of k_argmax_step and
// (with embed) the next token's embedding row into x; without, out_tokens[0]
struct StepIO {
  int* ctl;
  int* hist;
  int* out_tokens;
  const float* embed;
  int dm;
  float* x;
};

constexpr int kCandLds = 512;      // candidates kept in LDS when they fit
constexpr int kListsPerWave = kFront / (kThreads / 64);

constexpr int kSortMax = 4096;  // entries sorted in LDS by the draw without top-k
constexpr int kRankMax = 256;   // of them, by rank instead of a bitonic network

struct Smem {
  union {
    unsigned radix[16 * kThreads];  // sort_large: per-thread digit counts, then offsets
    uint64_t keys[kSortMax];        // draw_parallel: (~probability bits, id), ascending
  };
  double dscan[kThreads / 64];
  double dwork[4];
  Cand stage[kStage];
  Cand cand[kCandLds];
  Cand sel[kPartial];
  Cand sorted[kPartial];
  unsigned scan[kThreads];
  float fred[kThreads / 64];
  int ired[kThreads / 64];
  int iwork[8];
  float fwork[8];
};

__device__ __forceinline__ uint64_t rng_next(uint64_t& s) {
  uint64_t x = s;
  x ^= x >> 12;
  x ^= x << 25;
  x ^= x >> 27;
  s = x;
  return x * 0x2545F4914F6CDD1DULL;
}

__device__ __forceinline__ float rng_float(uint64_t& s) {
  return __fmul_rn((float)(rng_next(s) >> 11), 1.0f / 9007199254740992.0f);
}

// (int)f as x86-64 cvttss2si computes it
__device__ __forceinline__ int cvtt_x86(float f) {
  return (f >= -2147483648.0f && f < 2147483648.0f) ? (int)f : (int)0x80000000;
}

// max of n partial maxima under `x > m` from -1e30f; called by whole waves
__device__ __forceinline__ float front_max(const float* __restrict__ pmax, int n) {
  const int lane = threadIdx.x & 63;
  float v = -1e30f;
  // the first 8 * 64 maxima in one round of loads (indices clamped,
  // unconditional: loads in the loop would each wait for the one before)
  constexpr int FU = 8;
  float w[FU];
#pragma unroll
  for (int u = 0; u < FU; ++u) w[u] = pmax[min(lane + 64 * u, n - 1)];
#pragma unroll
  for (int u = 0; u < FU; ++u)
    if (lane + 64 * u < n && w[u] > v) v = w[u];
  for (int i = lane + 64 * FU; i < n; i += 64) {
    const float x = pmax[i];
    if (x > v) v = x;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float w = __shfl_xor(v, o, 64);
    if (w > v) v = w;
  }
  return __shfl(v, 0, 64);
}

// min_p threshold before the softmax (src/model.c:168-176)
__device__ __forceinline__ float min_p_threshold(float max_logit, float min_p) {
  if (min_p >= 1.0f) return max_logit;
  if (min_p > 0.0f) return __fadd_rn(max_logit, libm::logf_glibc(min_p));
  return -1e30f;
}

__host__ __device__ __forceinline__ int effective_k(int top_k) {
  return (top_k > 0 && top_k <= 256) ? top_k : 0;  // src/model.c:168-170
}

// Without top-k: whether draw_parallel is tried.  Not where min_p alone cuts
// (top_p >= 1): it leaves few candidates, which one thread walks in 16 us per
// call, 19 with the probabilities' launch and the buckets; for the same reason
// not for small vocabularies at top_p >= 1 (V = 64: 17.3 us, 18.9 tried; 256: 30.7,
// 19.0); and not where a top_k above 256 alone cuts, which only the full sort
// decides.
__host__ __device__ __forceinline__ bool tries_parallel(const SampleParams& p, int V) {
  return p.top_p < 1.0f || (!(p.min_p > 0.0f) && V >= 96 && (p.top_k <= 0 || p.top_k >= V));
}

__device__ __forceinline__ float bucket_scale_of() {
  return cr_divf((float)(kBuckets - 1), 20.0f);  // src/model.c:182
}

// extraction threshold for a cutoff bucket (src/model.c:208-213).  It does
// not increase with the cutoff, so cutoff kBuckets-1 gives the lowest.
__device__ __forceinline__ float extract_threshold(float max_logit, float min_p_thresh,
                                                   int cutoff) {
  const float bucket_thresh =
      __fsub_rn(max_logit, cr_divf((float)(cutoff + 1), bucket_scale_of()));
  return bucket_thresh > min_p_thresh ? bucket_thresh : min_p_thresh;
}

// p[i..i+3] with zeros at and past `end`; p is 16-byte aligned, i % 4 == 0
__device__ __forceinline__ float4 load4(const float* __restrict__ p, int i, int end) {
  if (i + 4 <= end) return *(const float4*)(p + i);
  float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (i < end) r.x = p[i];
  if (i + 1 < end) r.y = p[i + 1];
  if (i + 2 < end) r.z = p[i + 2];
  return r;
}

__device__ __forceinline__ void heap_sift_down(Cand* h, int n, int i) {
  while (true) {
    int smallest = i;
    const int l = 2 * i + 1, r = 2 * i + 2;
    if (l < n && h[l].val < h[smallest].val) smallest = l;
    if (r < n && h[r].val < h[smallest].val) smallest = r;
    if (smallest == i) break;
    const Cand t = h[i];
    h[i] = h[smallest];
    h[smallest] = t;
    i = smallest;
  }
}

// block-wide max of v under `x > m` from -1e30f (NaN never wins)
__device__ float block_max(float v, Smem& sm) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float w = __shfl_xor(v, o, 64);
    if (w > v) v = w;
  }
  if (lane == 0) sm.fred[wave] = v;
  __syncthreads();
  float m = -1e30f;
  for (int w = 0; w < kThreads / 64; ++w)
    if (sm.fred[w] > m) m = sm.fred[w];
  __syncthreads();
  return m;
}

// exclusive scan of one count per thread; returns this thread's offset,
// total in *total
__device__ unsigned block_scan(unsigned c, Smem& sm, unsigned* total) {
  sm.scan[threadIdx.x] = c;
  __syncthreads();
  for (int o = 1; o < kThreads; o <<= 1) {
    const unsigned add = threadIdx.x >= (unsigned)o ? sm.scan[threadIdx.x - o] : 0u;
    __syncthreads();
    sm.scan[threadIdx.x] += add;
    __syncthreads();
  }
  const unsigned incl = sm.scan[threadIdx.x];
  *total = sm.scan[kThreads - 1];
  __syncthreads();
  return incl - c;
}

// the candidates (i, v) with v >= thr in ascending i, from the front
// blocks' pre-candidate lists (each in index order, the blocks' segments
// ascending; pc: this wave's list lengths).  Wave w takes lists
// kListsPerWave * w .. + kListsPerWave - 1 and writes after the waves before
// it: into sm.cand when they all fit, else to `spill`.  Returns the count,
// the array in *out.
__device__ int gather(const Scratch& sc, const int (&pc)[kListsPerWave], int seg, float thr,
                      Cand* spill, Cand** out, Smem& sm) {
  constexpr int NW = kThreads / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int cnt = 0;
  // the first 64 entries of every list in one round of loads (index 0 of
  // an empty list is in bounds: a segment holds at least 4), kept for the
  // second pass; the rest in turns
  Cand first[kListsPerWave];
#pragma unroll
  for (int j = 0; j < kListsPerWave; ++j)
    first[j] = (sc.pre + (size_t)(wave * kListsPerWave + j) * seg)[min(lane, max(pc[j], 1) - 1)];
#pragma unroll
  for (int j = 0; j < kListsPerWave; ++j) {
    const Cand* src = sc.pre + (size_t)(wave * kListsPerWave + j) * seg;
    cnt += lane < pc[j] && first[j].val >= thr;
    for (int i = lane + 64; i < pc[j]; i += 64) cnt += src[i].val >= thr;
  }
  cnt = wave_sum_i32(cnt);
  if (lane == 0) sm.ired[wave] = cnt;
  __syncthreads();
  int off = 0, total = 0;
  for (int w = 0; w < NW; ++w) {
    const int c = sm.ired[w];
    off += w < wave ? c : 0;
    total += c;
  }
  __syncthreads();
  Cand* dst = total <= kCandLds ? sm.cand : spill;
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int j = 0; j < kListsPerWave; ++j) {
    const Cand* src = sc.pre + (size_t)(wave * kListsPerWave + j) * seg;
    for (int i0 = 0; i0 < pc[j]; i0 += 64) {
      const int i = i0 + lane;
      Cand x{0, 0.0f};
      if (i0 == 0)
        x = first[j];
      else if (i < pc[j])
        x = src[i];
      const bool h = i < pc[j] && x.val >= thr;
      const uint64_t m = __ballot(h);
      if (h) dst[off + __popcll(m & below)] = x;
      off += __popcll(m);
    }
  }
  __syncthreads();
  *out = dst;
  return total;
}

// the sequential scan `best = 0, best_v = init; if (logits[i] > best_v) ...`
// over i = 0 .. V-1: init = logits[0] in the pruned-everything guards
// (src/model.c:225-233, 285-291), -1e9f in the greedy branch
// (src/model.c:144-154).  A later value wins only when strictly greater, so
// NaNs never win.  Returned to every thread.
__device__ int argmax_scan(const float* __restrict__ logits, int V, float init, Smem& sm) {
  float bv = init;
  int bi = 0;
  for (int i = threadIdx.x; i < V; i += kThreads) {
    const float v = logits[i];
    if (v > bv) {  // ascending i per thread: the first maximum stays
      bv = v;
      bi = i;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float ov = __shfl_xor(bv, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if (lane == 0) {
    sm.fred[wave] = bv;
    sm.ired[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; ++w)
      if (sm.fred[w] > bv || (sm.fred[w] == bv && sm.ired[w] < bi)) {
        bv = sm.fred[w];
        bi = sm.ired[w];
      }
    sm.iwork[0] = bi;
  }
  __syncthreads();
  const int best = sm.iwork[0];
  __syncthreads();
  return best;
}

// stable descending order of n <= kPartial candidates: src -> dst
__device__ void sort_small(const Cand* src, Cand* dst, int n) {
  const int i = threadIdx.x;
  if (i < n) {
    const float v = src[i].val;
    int r = 0;
    for (int j = 0; j < n; ++j) {
      const float w = src[j].val;
      r += (w > v) || (w == v && j < i);
    }
    dst[r] = src[i];
  }
  __syncthreads();
}

// key of a float for an ascending radix order that puts larger values first
__device__ __forceinline__ uint32_t desc_key(float v) {
  const uint32_t u = __float_as_uint(v);
  const uint32_t asc = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ~asc;
}

// stable descending sort of n candidates in global memory (LSD radix, 4-bit
// digits, each thread a contiguous run); the result ends in `a`
__device__ void sort_large(Cand* a, Cand* b, int n, Smem& sm) {
  unsigned* cnt = sm.radix;  // [16][kThreads]
  const int per = (n + kThreads - 1) / kThreads;
  const int i0 = threadIdx.x * per, i1 = min(n, i0 + per);
  Cand* src = a;
  Cand* dst = b;
  for (int shift = 0; shift < 32; shift += 4) {
    unsigned c[16];
#pragma unroll
    for (int d = 0; d < 16; ++d) c[d] = 0;
    for (int i = i0; i < i1; ++i) ++c[(desc_key(src[i].val) >> shift) & 15];
#pragma unroll
    for (int d = 0; d < 16; ++d) cnt[d * kThreads + threadIdx.x] = c[d];
    __syncthreads();
    // exclusive offsets in (digit, thread) order: thread t scans its 16
    // entries t*16 .. t*16+15 of the flattened array, then the partials
    unsigned part = 0;
    for (int e = 0; e < 16; ++e) part += cnt[threadIdx.x * 16 + e];
    unsigned total;
    unsigned base = block_scan(part, sm, &total);
    unsigned own[16];
    for (int e = 0; e < 16; ++e) own[e] = cnt[threadIdx.x * 16 + e];
    __syncthreads();
    // rewrite the counts as exclusive offsets
    for (int e = 0; e < 16; ++e) {
      cnt[threadIdx.x * 16 + e] = base;
      base += own[e];
    }
    __syncthreads();
    unsigned off[16];
#pragma unroll
    for (int d = 0; d < 16; ++d) off[d] = cnt[d * kThreads + threadIdx.x];
    for (int i = i0; i < i1; ++i) {
      const Cand x = src[i];
      const int d = (desc_key(x.val) >> shift) & 15;
      dst[off[d]++] = x;
    }
    __syncthreads();
    Cand* t = src;
    src = dst;
    dst = t;
  }
  // 8 passes: the sorted run is back in `a`
}

// filter_and_sample (src/model.c:67-127) with min_p = 0.  Its three walks
// over c (top_p cut, renormalising sum, CDF) are sequential in the
// reference's order on thread 0; the block stages c through LDS.  The token
// is valid in thread 0.
__device__ int filter_and_sample(const Cand* __restrict__ c, int n, float top_p, int top_k,
                                 uint64_t& rng, Smem& sm) {
  // stage chunk [c0, c0 + m) of c into sm.stage
  auto stage = [&](int c0, int m) __attribute__((always_inline)) {
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += kThreads) sm.stage[i] = c[c0 + i];
    __syncthreads();
  };
  if (top_p < 1.0f) {
    double cs = 0.0;
    int cut = n;
    for (int c0 = 0; c0 < n; c0 += kStage) {
      const int m = min(kStage, n - c0);
      stage(c0, m);
      if (threadIdx.x == 0 && cut == n)
        for (int i = 0; i < m; ++i) {
          cs += (double)sm.stage[i].val;
          if (cs >= (double)top_p) {
            cut = c0 + i + 1;
            break;
          }
        }
      if (threadIdx.x == 0) sm.iwork[2] = cut;
      __syncthreads();
      cut = sm.iwork[2];
      if (cut != n) break;
    }
    n = cut;
  }
  if (top_k > 0 && top_k < n) n = top_k;
  double new_sum = 0.0;
  for (int c0 = 0; c0 < n; c0 += kStage) {
    const int m = min(kStage, n - c0);
    stage(c0, m);
    if (threadIdx.x == 0)
      for (int i = 0; i < m; ++i) new_sum += (double)sm.stage[i].val;
  }
  float r = 0.0f;
  if (threadIdx.x == 0) r = __fmul_rn(rng_float(rng), (float)new_sum);
  double cdf = 0.0;
  int token = -1;
  for (int c0 = 0; c0 < n; c0 += kStage) {
    const int m = min(kStage, n - c0);
    stage(c0, m);
    if (threadIdx.x == 0)
      for (int i = 0; i < m; ++i) {
        cdf += (double)sm.stage[i].val;
        if ((double)r < cdf) {
          token = sm.stage[i].id;
          break;
        }
      }
    if (threadIdx.x == 0) sm.iwork[3] = token;
    __syncthreads();
    token = sm.iwork[3];
    if (token >= 0) break;
  }
  if (token < 0) {
    stage(n - 1, 1);
    token = sm.stage[0].id;
  }
  __syncthreads();
  return token;
}

// the entries of c[0..m) (m <= kStage) whose value is above `root`, in
// order, into sm.stage; returns their count.  Wave w takes entries
// 256w .. 256w+255, four per lane.
__device__ int stage_above(const Cand* __restrict__ c, int m, float root, Smem& sm) {
  constexpr int NW = kThreads / 64, PER = kStage / NW;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  Cand x[PER / 64];
  uint64_t mk[PER / 64];
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < PER / 64; ++j) {
    const int i = wave * PER + 64 * j + lane;
    bool h = false;
    if (i < m) {
      x[j] = c[i];
      h = x[j].val > root;
    }
    mk[j] = __ballot(h);
    cnt += __popcll(mk[j]);
  }
  if (lane == 0) sm.ired[wave] = cnt;
  __syncthreads();
  int off = 0, total = 0;
  for (int w = 0; w < NW; ++w) {
    const int cw = sm.ired[w];
    off += w < wave ? cw : 0;
    total += cw;
  }
#pragma unroll
  for (int j = 0; j < PER / 64; ++j) {
    if ((mk[j] >> lane) & 1ull) sm.stage[off + __popcll(mk[j] & below)] = x[j];
    off += __popcll(mk[j]);
  }
  __syncthreads();
  return total;
}

// min-heap selection of the k largest of c[0..n) (src/model.c:238-250,
// 322-337), one thread; c is global memory, staged through LDS.  The root
// never decreases (a replacement is larger than the old root, and after the
// sift the root is the replacement or a child that was not below the old
// root), so entries not above the root when their chunk is staged would be
// passed over and are not staged.
__device__ void heap_select(const Cand* __restrict__ c, int n, int k, Cand* heap, Smem& sm) {
  for (int i = threadIdx.x; i < k; i += kThreads) heap[i] = c[i];
  __syncthreads();
  if (threadIdx.x == 0)
    for (int i = k / 2 - 1; i >= 0; --i) heap_sift_down(heap, k, i);
  for (int c0 = k; c0 < n; c0 += kStage) {
    const int m = min(kStage, n - c0);
    __syncthreads();
    const int kept = stage_above(c + c0, m, heap[0].val, sm);
    if (threadIdx.x == 0)
      for (int i = 0; i < kept; ++i)
        if (sm.stage[i].val > heap[0].val) {
          heap[0] = sm.stage[i];
          heap_sift_down(heap, k, 0);
        }
  }
  __syncthreads();
}

// sum of (double) c[0..n).val in order, one thread, staged through LDS
__device__ double ordered_sum(const Cand* __restrict__ c, int n, Smem& sm) {
  double s = 0.0;
  for (int c0 = 0; c0 < n; c0 += kStage) {
    const int m = min(kStage, n - c0);
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += kThreads) sm.stage[i] = c[c0 + i];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int i = 0; i < m; ++i) s += (double)sm.stage[i].val;
  }
  __syncthreads();
  return s;
}

// the generator state back, then the step bookkeeping of k_argmax_step
// (or, without ctl, the token alone); one thread
// the step counters, read by thread 0 when the kernel starts (nothing else
// in the step writes them) so that the bookkeeping at its end waits for no
// load
struct CtlSnap {
  int step = 0, hcount = 0, pos = 0, done = 0;
};
__device__ __forceinline__ CtlSnap ctl_snap(const StepIO& io) {
  CtlSnap c;
  if (threadIdx.x == 0 && io.ctl) {
    c.step = io.ctl[kCtlStep];
    c.hcount = io.ctl[kCtlHcount];
    c.pos = io.ctl[kCtlPos];
    c.done = io.ctl[kCtlDone];
  }
  return c;
}

__device__ void finish_step(int token, uint64_t rng, uint64_t* rng_state, const StepIO& io,
                            const CtlSnap& c) {
  *rng_state = rng;
  if (!io.ctl) {
    io.out_tokens[0] = token;
    return;
  }
  int* ctl = io.ctl;
  if (io.out_tokens) io.out_tokens[c.step] = token;
  ctl[kCtlStep] = c.step + 1;
  ctl[kCtlToken] = token;
  io.hist[c.hcount % kHist] = token;
  ctl[kCtlHcount] = c.hcount + 1;
  ctl[kCtlPos] = c.pos + 1 < 3 ? c.pos + 1 : 0;  // src/block.c:107
  if (c.done == kDoneArmed && (token == 50256 || token == 0)) ctl[kCtlDone] = kDoneStopped;
}

// the next token's embedding row (src/model.c:1116-1122), whole block
__device__ void embed_next(int token, const StepIO& io) {
  if (!io.ctl || !io.embed) return;
  const float* __restrict__ row = io.embed + (size_t)token * io.dm;
  for (int i = threadIdx.x; i < io.dm; i += kThreads) io.x[i] = row[i];
}

// ---------------------------------------------------------------------------
// The draw without top-k (src/model.c:278-361) from sums in any order.
//
// The reference adds probabilities one by one in double, and only decisions
// and fp32 roundings of those sums reach its result.  A double sum of n
// non-negative terms is within (n - 1) 2^-53 of the exact one, relative,
// whatever the order; so where a sum of the same terms in another order, widened
// by twice that and more (sum_slack), decides or rounds the same way at both
// ends, the reference's does too.  Where it does not, the sum may still be exact
// in every order (exact_sum, bm_exact.h): sums of few terms are, and they often
// lie on the midpoint of two floats, or on top_p itself; that is looked into
// only then.  Where neither says (the sum over a large vocabulary close to a
// rounding, about n 2^-26 of the draws), or where the drawn token's probability
// is tied in the min-heap's order, draw_parallel returns false and the
// sequential code below runs.  So does it where more than kSortMax entries share
// the bucket that decides, and for a top_k that cuts (above 256).  Of 200 vectors
// of spread 4 at temp = 0.8, top_p = 0.9, by the slack alone 31 went that way at
// V = 1000, min_p = 0.05 (9 at min_p = 0) and 14 at V = 50257, min_p = 0.05; none
// of them now.
// V = 50257, logits of spread 4 at temp = 0.8, top_p = 0.9: 2759 us per call
// in turn on one thread (the sum, then the heap), 48 us this way (52 with LDS
// shuffles in the scans, 55.9 with a bitonic network for any count too).
// ---------------------------------------------------------------------------
// prefix sums over the wave on DPP (a shuffle through LDS per step costs
// several times as much)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double v) {  // lanes without a source get 0
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)dpp_or0<CTRL, ROWS>((int)(uint32_t)u);
  const uint32_t hi = (uint32_t)dpp_or0<CTRL, ROWS>((int)(uint32_t)(u >> 32));
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ __forceinline__ double wave_scan_f64(double v) {
  v += dpp_f64<0x111, 0xf>(v);
  v += dpp_f64<0x112, 0xf>(v);
  v += dpp_f64<0x114, 0xf>(v);
  v += dpp_f64<0x118, 0xf>(v);
  v += dpp_f64<0x142, 0xa>(v);
  return v + dpp_f64<0x143, 0xc>(v);
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ __forceinline__ double wave_sum_f64(double v) { return lane_f64(wave_scan_f64(v), 63); }

// every thread has the same v: make the branches on it uniform (barriers
// follow on both sides of them)
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ double sum_slack(double sum, int n) { return sum * (double)n * 0x1p-51; }

// (float)sum of the reference's sum, if every sum within the slack rounds alike
__device__ __forceinline__ bool sure_float(double sum, double slack, float* f) {
  *f = (float)(sum - slack);
  return uni(*f == (float)(sum + slack) && *f > 0.0f && *f < __builtin_inff());
}

// the wave's smallest v
__device__ __forceinline__ float wave_least(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return lane_f32(v, 0);
}

// block-wide inclusive prefix sum; *before = the sum in front of the thread
__device__ double block_scan_f64(double v, double* before, Smem& sm) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double incl = wave_scan_f64(v);
  __syncthreads();
  if (lane == 63) sm.dscan[wave] = incl;
  __syncthreads();
  double off = 0.0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {  // all loads at once
    const double t = sm.dscan[w];
    off += w < wave ? t : 0.0;
  }
  *before = off + dpp_f64<0x138, 0xf>(incl);
  return off + incl;
}

// the listed probabilities of buckets lo..hi (at most kSortMax), as sorted
// keys in sm.keys; returns their count
__device__ int sort_buckets(const Scratch& sc, const int (&pc)[kListsPerWave], int seg, int lo,
                            int hi, Smem& sm) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  __syncthreads();
  if (threadIdx.x == 0) sm.iwork[6] = 0;
  __syncthreads();
  constexpr int U = 4;  // 16-byte loads in flight per list
#pragma unroll
  for (int j = 0; j < kListsPerWave; ++j) {
    const size_t base = (size_t)(wave * kListsPerWave + j) * seg;
    for (int i0 = 0; i0 < pc[j]; i0 += 256 * U) {
      float4 q[U];
#pragma unroll
      for (int u = 0; u < U; ++u)  // a list has room for seg entries, a multiple of 4
        q[u] = *(const float4*)(sc.pv + base + min(i0 + 256 * u + 4 * lane, seg - 4));
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float v[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = i0 + 256 * u + 4 * lane + e;
          const int b = p_bucket(v[e]);
          const bool h = i < pc[j] && b >= lo && b <= hi;
          const uint64_t m = __ballot(h);
          if (!m) continue;
          int at = 0;
          if (lane == 0) at = atomicAdd(&sm.iwork[6], __popcll(m));
          at = __builtin_amdgcn_readfirstlane(at) + __popcll(m & below);
          if (h && at < kSortMax)
            sm.keys[at] = (uint64_t)~__float_as_uint(v[e]) << 32 | (uint32_t)sc.pre[base + i].id;
        }
      }
    }
  }
  __syncthreads();
  const int n = min(uni(sm.iwork[6]), kSortMax);
  if (n <= kRankMax) {  // few: each key's rank by comparing it with all
    uint64_t own = 0;
    int r = 0;
    if ((int)threadIdx.x < n) {
      own = sm.keys[threadIdx.x];
#pragma unroll 4
      for (int i = 0; i < n; ++i) r += sm.keys[i] < own;
    }
    __syncthreads();
    if ((int)threadIdx.x < n) sm.keys[r] = own;
    __syncthreads();
    return n;
  }
  int size = 64;
  while (size < n) size *= 2;
  for (int i = n + threadIdx.x; i < size; i += kThreads) sm.keys[i] = ~0ull;
  // bitonic: larger probabilities first, equal ones by ascending id
  for (int k = 2; k <= size; k *= 2)
    for (int d = k / 2; d >= 1; d /= 2) {
      __syncthreads();
      for (int t = threadIdx.x; t < size / 2; t += kThreads) {
        const int i = 2 * t - (t & (d - 1)), l = i + d;
        const uint64_t a = sm.keys[i], b = sm.keys[l];
        if ((a > b) == ((i & k) == 0)) {
          sm.keys[i] = b;
          sm.keys[l] = a;
        }
      }
    }
  __syncthreads();
  return n;
}

__device__ __forceinline__ float key_prob(uint64_t k) { return __uint_as_float(~(uint32_t)(k >> 32)); }

// first sorted entry whose running sum (from `base`, of larger terms) passes x
// -- is >= x (INCL) or > x -- and whether that is sure; the running sum there in
// *at.  first: nothing comes before entry 0.  n if none passes.
template <bool INCL>
__device__ int find_key(int n, double base, double x, double slack, bool first, bool* sure,
                        double* at, Smem& sm) {
  double v[kSortMax / kThreads], own = 0.0, before;
  const int i0 = threadIdx.x * (kSortMax / kThreads);
#pragma unroll
  for (int e = 0; e < kSortMax / kThreads; ++e) {
    v[e] = i0 + e < n ? (double)key_prob(sm.keys[i0 + e]) : 0.0;
    own += v[e];
  }
  block_scan_f64(own, &before, sm);
  if (threadIdx.x == 0) sm.iwork[7] = n;
  __syncthreads();
  double run = base + before;
  bool found = false;
#pragma unroll
  for (int e = 0; e < kSortMax / kThreads; ++e) {
    run += v[e];
    if (!found && i0 + e < n && (INCL ? run >= x : run > x)) {
      found = true;
      atomicMin(&sm.iwork[7], i0 + e);
    }
  }
  __syncthreads();
  const int j = uni(sm.iwork[7]);
  if (j < n && j >= i0 && j < i0 + kSortMax / kThreads) {
    double r = base + before;
#pragma unroll
    for (int e = 0; e < kSortMax / kThreads; ++e)
      if (i0 + e <= j) {
        sm.dwork[1] = r;
        r += v[e];
      }
    sm.dwork[0] = r;
  }
  __syncthreads();
  *at = sm.dwork[0];
  *sure = uni(j < n && sm.dwork[0] > x + slack && ((first && j == 0) || sm.dwork[1] < x - slack));
  if (__builtin_expect(!*sure && uni(j < n), 0))  // every term so far is at least entry j's
    *sure = uni(exact_sum(sm.dwork[0], key_prob(sm.keys[j])) &&
                ((first && j == 0) || (INCL ? sm.dwork[1] < x : sm.dwork[1] <= x)));
  __syncthreads();
  return j;
}

// first bucket, from the largest probabilities down, whose running sum
// passes x; in front of it: *sum and *cnt.  -1 if none passes.
template <bool INCL>
__device__ int find_bucket(const double (&s)[2], const int (&c)[2], double x, double* sum, int* cnt,
                           Smem& sm) {
  // counts below 2^53 add exactly as doubles
  double sb, cb_d;
  block_scan_f64(s[0] + s[1], &sb, sm);
  block_scan_f64((double)(c[0] + c[1]), &cb_d, sm);
  const int cb = (int)cb_d;
  if (threadIdx.x == 0) sm.iwork[7] = kPBuckets;
  __syncthreads();
  const double r0 = sb + s[0], r1 = r0 + s[1];
  const int d = 2 * threadIdx.x;
  if (c[0] && (INCL ? r0 >= x : r0 > x))
    atomicMin(&sm.iwork[7], d);
  else if (c[1] && (INCL ? r1 >= x : r1 > x))
    atomicMin(&sm.iwork[7], d + 1);
  __syncthreads();
  const int at = uni(sm.iwork[7]);
  if (at == d || at == d + 1) {
    sm.dwork[2] = at == d ? sb : r0;
    sm.iwork[5] = at == d ? cb : cb + c[0];
  }
  __syncthreads();
  *sum = sm.dwork[2];
  *cnt = uni(sm.iwork[5]);
  __syncthreads();
  return at == kPBuckets ? -1 : kPBuckets - 1 - at;
}

// the smallest listed probability that is not zero
__device__ float least_prob(const Scratch& sc, const int (&pc)[kListsPerWave], int seg, Smem& sm) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float v = __builtin_inff();
  for (int j = 0; j < kListsPerWave; ++j) {
    const float* __restrict__ list = sc.pv + (size_t)(wave * kListsPerWave + j) * seg;
    for (int i = lane; i < pc[j]; i += 64)
      if (list[i] > 0.0f) v = fminf(v, list[i]);
  }
  v = wave_least(v);
  __syncthreads();
  if (lane == 0) sm.fred[wave] = v;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) v = fminf(v, sm.fred[w]);
  __syncthreads();
  return v;
}

__device__ bool draw_parallel(const Scratch& sc, const int (&pc)[kListsPerWave], int seg,
                              const SampleParams& p, uint64_t& rng, int* token, Smem& sm) {
  static_assert(kFront == 64 && kPBuckets == 2 * kThreads, "lane / thread per list / buckets");
  const int lane = threadIdx.x & 63;
  const int mine = sc.pcnt[lane];
  const int n = wave_sum_i32(mine);
  float f;
  const int scaled = *sc.scaled;  // looked at once the sums have arrived too
  const double ps = sc.psum[lane], total = wave_sum_f64(ps);
  const double slack = sum_slack(total, n);
  auto total_sure = [&](float* v) {  // (float)total
    return sure_float(total, slack, v) ||
           (uni(exact_sum(total, least_prob(sc, pc, seg, sm))) && sure_float(total, 0.0, v));
  };
  if (!uni(scaled)) return false;
  uint64_t g = rng;
  if (p.top_p >= 1.0f && (p.top_k <= 0 || p.top_k >= n)) {
    // in index order: the list, then the entry the walk ends at
    if (!total_sure(&f)) return false;
    const double r = (double)__fmul_rn(rng_float(g), f);
    const double incl = wave_scan_f64(ps);
    const uint64_t hit = __ballot(mine > 0 && incl > r);
    if (!hit) return false;
    const int l = __ffsll((unsigned long long)hit) - 1;
    const double base = l ? lane_f64(incl, l - 1) : 0.0;
    const int cnt = __builtin_amdgcn_readlane(mine, l);
    const size_t at = (size_t)l * seg;
    static_assert(kMaxVocab / kFront + 4 <= 4 * kThreads, "a list fits one pass");
    double v[4], own = 0.0, before;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * threadIdx.x + e;
      v[e] = i < cnt ? (double)sc.pv[at + i] : 0.0;
      own += v[e];
    }
    block_scan_f64(own, &before, sm);
    if (threadIdx.x == 0) sm.iwork[7] = -1;
    __syncthreads();
    double run = base + before;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * threadIdx.x + e;
      const double next = run + v[e];
      if (next > r + slack && (run < r - slack || (l == 0 && i == 0)))  // one entry at most
        sm.iwork[7] = sc.pre[at + min(i, seg - 1)].id;
      run = next;
    }
    __syncthreads();
    *token = uni(sm.iwork[7]);
    __syncthreads();
    if (*token < 0) return false;
    rng = g;
    return true;
  }
  if (p.top_p >= 1.0f) return false;  // top_k > 256 alone: by the sort

  // sorted: the cut at top_p
  double s[2];
  int c[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int b = kPBuckets - 1 - 2 * (int)threadIdx.x - e;
    s[e] = sc.bsum[b];
    c[e] = sc.bcnt[b];
  }
  const double tp = (double)p.top_p;
  double front = 0.0, kept;
  int fcnt = 0, ncut = n, held = -1, n_held = 0;  // held: the bucket(s) in sm.keys
  bool all = false, sure;
  const int bc = find_bucket<true>(s, c, tp, &front, &fcnt, sm);
  auto count_of = [&](int b) {  // the bucket's count, to every thread
    const int t = (kPBuckets - 1 - b) / 2, e = (kPBuckets - 1 - b) & 1;
    if ((int)threadIdx.x == t) sm.iwork[6] = e ? c[1] : c[0];
    __syncthreads();
    const int r = uni(sm.iwork[6]);
    __syncthreads();
    return r;
  };
  if (bc < 0) {
    if (uni(total + slack >= tp) || !total_sure(&f)) return false;
  } else {
    const int cnt = count_of(bc);
    all = fcnt + cnt <= kSortMax;
    if (!all && cnt > kSortMax) return false;
    if (all) front = 0.0, fcnt = 0;
    n_held = sort_buckets(sc, pc, seg, bc, all ? kPBuckets - 1 : bc, sm);
    held = bc;
    const int j = find_key<true>(n_held, front, tp, slack, fcnt == 0, &sure, &kept, sm);
    if (!sure) return false;
    ncut = fcnt + j + 1;
    // every term is at least the last one
    if (!sure_float(kept, sum_slack(kept, ncut), &f) &&
        !(uni(exact_sum(kept, key_prob(sm.keys[j]))) && sure_float(kept, 0.0, &f)))
      return false;
  }
  if (p.top_k > 0 && p.top_k < ncut) return false;
  const double r = (double)__fmul_rn(rng_float(g), f);
  if (!all) {
    const int br = find_bucket<false>(s, c, r, &front, &fcnt, sm);
    if (br < 0) return false;
    if (br != held) {
      if (count_of(br) > kSortMax) return false;
      n_held = sort_buckets(sc, pc, seg, br, br, sm);
    }
  }
  const int j = find_key<false>(n_held, front, r, slack, fcnt == 0, &sure, &kept, sm);
  if (!sure || fcnt + j >= ncut) return false;
  const uint64_t key = sm.keys[j];
  // up to kPartial entries come out of the min-heap, whose order decides
  // among equal ones; a full sort keeps them by index
  if (n > kPartial && ncut <= kPartial) {
    const uint32_t hi = (uint32_t)(key >> 32);
    if (uni((j > 0 && (uint32_t)(sm.keys[j - 1] >> 32) == hi) ||
            (j + 1 < n_held && (uint32_t)(sm.keys[j + 1] >> 32) == hi)))
      return false;
  }
  *token = uni((int)(uint32_t)key);
  rng = g;
  return true;
}

}  // namespace

// Front pass 1: logits[i] *= 1/temp over the block's segment and the
// segment's max under `x > m` from -1e30f (src/model.c:160-166).  Block 0
// also clears the histogram.  (The LM head can do this pass itself, with its
// own blocks' maxima.)
__global__ __launch_bounds__(kFrontThreads) void k_samp_scale(float* __restrict__ logits, int V,
                                                              float temp, void* scratch,
                                                              const int* ctl) {
  __shared__ float red[kFrontThreads / 64];
  if (step_stopped(ctl)) return;
  const Scratch sc = scratch_of(scratch, V);
  const int seg = front_seg(V);
  const int i0 = min(V, (int)blockIdx.x * seg), i1 = min(V, i0 + seg);
  if (blockIdx.x == 0 && threadIdx.x < kBuckets) sc.hist[threadIdx.x] = 0;
  const float inv_temp = cr_divf(1.0f, temp);
  float mx = -1e30f;
  for (int i = i0 + 4 * (int)threadIdx.x; i < i1; i += 4 * kFrontThreads) {
    const float4 q = load4(logits, i, i1);
    float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = __fmul_rn(v[e], inv_temp);
      if (i + e < i1 && v[e] > mx) mx = v[e];
    }
    if (i + 4 <= i1) {
      *(float4*)(logits + i) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < i1) logits[i + e] = v[e];
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float w = __shfl_xor(mx, o, 64);
    if (w > mx) mx = w;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kFrontThreads / 64; ++w)
      if (red[w] > mx) mx = red[w];
    sc.pmax[blockIdx.x] = mx;
  }
}

// Front pass 2, kFront blocks: with the global max (of the npart partial
// maxima in pmax), each block writes its segment's pre-candidates: (i,
// logits[i]) with logits[i] >= the lowest extraction threshold, in index
// order, to pre[block * seg ..].
// TOPK: it also adds the segment's counts to the 128-bucket histogram over
// logits >= the min_p threshold (src/model.c:180-194).  PAR (tries_parallel):
// it also writes exp(logit - max) of the candidates to pv and their sum to
// esum.  Neither (min_p alone, say): the pre-candidates only.
template <bool TOPK, bool PAR>
__global__ __launch_bounds__(kFrontThreads) void k_samp_hist(const float* __restrict__ logits,
                                                             int V, SampleParams p,
                                                             void* scratch,
                                                             const float* __restrict__ pmax,
                                                             int npart, const int* ctl) {
  constexpr int NW = kFrontThreads / 64;
  __shared__ int bhist[kBuckets];
  __shared__ int wcnt[NW];
  if (step_stopped(ctl)) return;
  const Scratch sc = scratch_of(scratch, V);
  const int seg = front_seg(V);
  const int i0 = min(V, (int)blockIdx.x * seg), i1 = min(V, i0 + seg);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float4 q = load4(logits, i0 + 4 * (int)threadIdx.x, i1);  // before the max: independent
  const float max_logit = front_max(pmax, npart);
  const float min_p_thresh = min_p_threshold(max_logit, p.min_p);
  constexpr bool use_hist = TOPK;
  constexpr bool exps = !TOPK && PAR;  // tries_parallel
  const float bucket_scale = bucket_scale_of();
  const float pre_thresh =
      use_hist ? extract_threshold(max_logit, min_p_thresh, kBuckets - 1) : min_p_thresh;
  if (threadIdx.x < kBuckets) bhist[threadIdx.x] = 0;
  __shared__ double wsum[NW];
  // k_samp_probs adds to the buckets after this kernel
  constexpr int kClear = kPBuckets / kFront;
  if (exps && threadIdx.x < kClear) {
    sc.bsum[blockIdx.x * kClear + threadIdx.x] = 0.0;
    sc.bcnt[blockIdx.x * kClear + threadIdx.x] = 0;
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
  Cand* pre = sc.pre + (size_t)blockIdx.x * seg;
  float* pv = sc.pv + (size_t)blockIdx.x * seg;
  double esum = 0.0;
  int last = 0, off = 0;
  // the segment in rows of 4 * kFrontThreads entries (one row up to 65536
  // vocabulary entries), each compacted in index order after the last
  for (int i = i0 + 4 * (int)threadIdx.x, first = 1; i - 4 * (int)threadIdx.x < i1;
       i += 4 * kFrontThreads, first = 0) {
    const float4 qr = first ? q : load4(logits, i, i1);
    const float v[4] = {qr.x, qr.y, qr.z, qr.w};
    bool h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = i + e < i1;
      if (use_hist && in && v[e] >= min_p_thresh) {
        int b = cvtt_x86(__fmul_rn(__fsub_rn(max_logit, v[e]), bucket_scale));
        if (b >= kBuckets) b = kBuckets - 1;
        if (b < 0) b = 0;
        // the last bucket (20 or more below the max) takes most of the
        // vocabulary without a min_p threshold: counted in a register
        if (b == kBuckets - 1)
          ++last;
        else
          atomicAdd(&bhist[b], 1);
      }
      h[e] = in && v[e] >= pre_thresh;
    }
    // order-preserving compaction: lanes in order, then the waves
    uint64_t m[4];
    int wn = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      m[e] = __ballot(h[e]);
      wn += __popcll(m[e]);
    }
    if (lane == 0) wcnt[wave] = wn;
    __syncthreads();
    int base = off, row = 0;
    for (int w = 0; w < NW; ++w) {
      base += w < wave ? wcnt[w] : 0;
      row += wcnt[w];
    }
    __syncthreads();
    int pos = base;
#pragma unroll
    for (int e = 0; e < 4; ++e) pos += __popcll(m[e] & below);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (h[e]) {
        if (exps) {  // the softmax numerator (src/model.c:292-297)
          const float ex = libm::expf_glibc(__fsub_rn(v[e], max_logit));
          pv[pos] = ex;
          esum += (double)ex;
        }
        pre[pos++] = Cand{i + e, v[e]};
      }
    off += row;
  }
  if (exps) {
    esum = wave_sum_f64(esum);
    if (lane == 0) wsum[wave] = esum;
    __syncthreads();
    if (threadIdx.x == 0) sc.esum[blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
  }
  if (use_hist) {
    last = wave_sum_i32(last);
    if (lane == 0 && last) atomicAdd(&bhist[kBuckets - 1], last);
    __syncthreads();
    if (threadIdx.x < kBuckets && bhist[threadIdx.x])
      atomicAdd(&sc.hist[threadIdx.x], bhist[threadIdx.x]);
  }
  if (threadIdx.x == 0) sc.pcnt[blockIdx.x] = off;
}

// Front pass 3 (PAR), kFront blocks: the probabilities pv * 1/sum, their
// sum per block, and the count and sum of each value bucket over all blocks.
__global__ __launch_bounds__(kFrontThreads) void k_samp_probs(int V, void* scratch,
                                                              const int* ctl) {
  __shared__ double bsum[kPBuckets];
  __shared__ int bcnt[kPBuckets];
  __shared__ double wsum[kFrontThreads / 64];
  __shared__ float wlo[kFrontThreads / 64], whi[kFrontThreads / 64];
  static_assert(kFrontThreads == 256, "four waves");
  if (step_stopped(ctl)) return;
  const Scratch sc = scratch_of(scratch, V);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, cnt = sc.pcnt[blockIdx.x];
  // 1 / (float)sum (src/model.c:298)
  const int n = uni(wave_sum_i32(sc.pcnt[lane]));
  const double esum = wave_sum_f64(sc.esum[lane]);
  for (int b = threadIdx.x; b < kPBuckets; b += kFrontThreads) {
    bsum[b] = 0.0;
    bcnt[b] = 0;
  }
  float f;
  bool ok = n > 0 && sure_float(esum, sum_slack(esum, n), &f);
  if (__builtin_expect(n > 0 && !ok, 0)) {
    // exact?  The smallest numerator from the smallest candidate, halved: expf
    // is monotone but for its last bit
    float lo = __builtin_inff(), hi = -__builtin_inff();
    for (int l = 0; l < kFront; ++l) {
      const Cand* __restrict__ list = sc.pre + (size_t)l * front_seg(V);
      for (int i = threadIdx.x; i < sc.pcnt[l]; i += kFrontThreads) {
        lo = fminf(lo, list[i].val);
        hi = fmaxf(hi, list[i].val);
      }
    }
    lo = wave_least(lo);
    hi = -wave_least(-hi);
    if (lane == 0) {
      wlo[wave] = lo;
      whi[wave] = hi;
    }
    __syncthreads();
    lo = fminf(fminf(wlo[0], wlo[1]), fminf(wlo[2], wlo[3]));
    hi = fmaxf(fmaxf(whi[0], whi[1]), fmaxf(whi[2], whi[3]));
    const float least = 0.5f * libm::expf_glibc(__fsub_rn(lo, hi));
    ok = uni(exact_sum(esum, least)) && sure_float(esum, 0.0, &f);
  }
  const float inv = ok ? cr_divf(1.0f, f) : 0.0f;
  if (blockIdx.x == 0 && threadIdx.x == 0) *sc.scaled = ok;
  __syncthreads();
  if (!ok) return;  // k_sample takes the sequential path
  float* pv = sc.pv + (size_t)blockIdx.x * front_seg(V);
  double sum = 0.0;
  for (int i = threadIdx.x; i < cnt; i += kFrontThreads) {
    const float v = __fmul_rn(pv[i], inv);
    pv[i] = v;
    sum += (double)v;
    const int b = p_bucket(v);
    atomicAdd(&bcnt[b], 1);
    unsafeAtomicAdd(&bsum[b], (double)v);
  }
  sum = wave_sum_f64(sum);
  if (lane == 0) wsum[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) sc.psum[blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
  for (int b = threadIdx.x; b < kPBuckets; b += kFrontThreads)
    if (bcnt[b]) {
      atomicAdd(&sc.bcnt[b], bcnt[b]);
      unsafeAtomicAdd(&sc.bsum[b], bsum[b]);
    }
}

// The rest of sample_advanced on one 1024-thread block, after the front
// passes: the cutoff bucket, the candidates filtered from the pre-candidate
// lists in order, selection, softmax, sorting and the draw; then the step
// bookkeeping and the next token's embedding (StepIO).  Leaves the
// histogram cleared for the next call.
// TOPK: an effective top-k; PAR: without one, tries_parallel.  Separate
// kernels, since the ways share little and the largest one's registers cost
// the others ~2 of 16 to 20 us per call.
template <bool TOPK, bool PAR>
__global__ __launch_bounds__(1024) void k_sample(const float* __restrict__ logits, int V,
                                                 SampleParams p, uint64_t* __restrict__ rng_state,
                                                 void* scratch, const float* __restrict__ pmax,
                                                 int npart, StepIO io) {
  __shared__ Smem sm;
  const Scratch sc = scratch_of(scratch, V);
  const int seg = front_seg(V);
  // every load that does not depend on another goes out first
  const CtlSnap cs = ctl_snap(io);
  const int wave = threadIdx.x >> 6;
  int hc0 = 0, hc1 = 0;
  if (threadIdx.x < 64) {
    hc0 = sc.hist[2 * threadIdx.x];
    hc1 = sc.hist[2 * threadIdx.x + 1];
  }
  int pc[kListsPerWave];
#pragma unroll
  for (int j = 0; j < kListsPerWave; ++j) pc[j] = sc.pcnt[wave * kListsPerWave + j];
  uint64_t rng = *rng_state;
  const float max_logit = front_max(pmax, npart);
  const float min_p_thresh = min_p_threshold(max_logit, p.min_p);
  int token = 0;
  Cand* probs = sc.probs;
  if constexpr (TOPK) {
    const int eff_k = effective_k(p.top_k);
    // the cutoff bucket (src/model.c:196-213): first bucket whose running
    // count reaches k; lane l of wave 0 holds buckets 2l, 2l+1
    if (threadIdx.x < 64) {
      const int l = threadIdx.x;
      const int c0 = hc0, c1 = hc1;
      int run = c0 + c1;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(run, o, 64);
        if (l >= o) run += up;
      }
      const int before = run - (c0 + c1);
      const bool at0 = before + c0 >= eff_k, at1 = !at0 && run >= eff_k;
      const uint64_t hit = __ballot(at0 || at1);
      int cutoff = kBuckets - 1;
      if (hit) {
        const int first = __ffsll((unsigned long long)hit) - 1;
        const int a0 = __shfl(at0 ? 1 : 0, first, 64);
        cutoff = 2 * first + (a0 ? 0 : 1);
      }
      if (l == 0) sm.fwork[0] = extract_threshold(max_logit, min_p_thresh, cutoff);
    }
    __syncthreads();
    const float extract_thresh = sm.fwork[0];
    int n = gather(sc, pc, seg, extract_thresh, sc.probs, &probs, sm);
    if (n == 0) {
      token = argmax_scan(logits, V, logits[0], sm);
    } else {
      // top-k by a min-heap when there are more candidates (src/model.c:236-251)
      if (n > eff_k) {
        heap_select(probs, n, eff_k, sm.sel, sm);
        n = eff_k;
      } else {
        for (int i = threadIdx.x; i < n; i += kThreads) sm.sel[i] = probs[i];
        __syncthreads();
      }
      // softmax on the survivors (src/model.c:253-266)
      float lm = -1e30f;
      if ((int)threadIdx.x < n) lm = sm.sel[threadIdx.x].val;
      const float local_max = block_max(lm, sm);
      if ((int)threadIdx.x < n)
        sm.sel[threadIdx.x].val = libm::expf_glibc(__fsub_rn(sm.sel[threadIdx.x].val, local_max));
      __syncthreads();
      if (threadIdx.x == 0) {
        double sum_exp = 0.0;
        for (int i = 0; i < n; ++i) sum_exp += (double)sm.sel[i].val;
        sm.fwork[1] = cr_divf(1.0f, (float)sum_exp);
      }
      __syncthreads();
      const float inv_sum = sm.fwork[1];
      if ((int)threadIdx.x < n) sm.sel[threadIdx.x].val = __fmul_rn(sm.sel[threadIdx.x].val, inv_sum);
      __syncthreads();
      const Cand* src = sm.sel;
      if (p.top_p < 1.0f) {  // src/model.c:268-274
        sort_small(sm.sel, sm.sorted, n);
        src = sm.sorted;
      }
      token = filter_and_sample(src, n, p.top_p, 0, rng, sm);
    }
  } else {
    bool drawn = false;
    if constexpr (PAR) drawn = draw_parallel(sc, pc, seg, p, rng, &token, sm);
    if (!drawn) {
      // no top-k: every candidate over the min_p threshold (src/model.c:278-300)
      Cand* probs2 = sc.pre;  // free once the candidates are gathered
      int n = gather(sc, pc, seg, min_p_thresh, sc.probs, &probs, sm);
      if (n == 0) {
        token = argmax_scan(logits, V, logits[0], sm);
      } else {
        for (int i = threadIdx.x; i < n; i += kThreads)
          probs[i].val = libm::expf_glibc(__fsub_rn(probs[i].val, max_logit));
        __syncthreads();
        const double sum_exp = ordered_sum(probs, n, sm);
        if (threadIdx.x == 0) sm.fwork[1] = cr_divf(1.0f, (float)sum_exp);
        __syncthreads();
        const float inv_sum = sm.fwork[1];
        for (int i = threadIdx.x; i < n; i += kThreads) probs[i].val = __fmul_rn(probs[i].val, inv_sum);
        __syncthreads();
        bool done = false;
        if (p.top_p >= 1.0f && (p.top_k <= 0 || p.top_k >= n)) {  // src/model.c:306-307
          // order-independent: the candidates stay in index order
          token = filter_and_sample(probs, n, p.top_p, p.top_k, rng, sm);
          done = true;
        }
        if (!done && p.top_p < 1.0f && n > kPartial) {  // src/model.c:313-343
          heap_select(probs, n, kPartial, sm.sel, sm);
          sort_small(sm.sel, sm.sorted, kPartial);
          if (threadIdx.x == 0) {
            double cs = 0.0;
            int hit = 0;
            for (int i = 0; i < kPartial; ++i) {
              cs += (double)sm.sorted[i].val;
              if (cs >= (double)p.top_p) {
                hit = 1;
                break;
              }
            }
            sm.iwork[1] = hit;
          }
          __syncthreads();
          done = sm.iwork[1] != 0;
          __syncthreads();
          if (done) {
            // sm.sorted is read through the staging buffer
            for (int i = threadIdx.x; i < kPartial; i += kThreads) sm.sel[i] = sm.sorted[i];
            __syncthreads();
            token = filter_and_sample(sm.sel, kPartial, p.top_p, p.top_k, rng, sm);
          }
        }
        if (!done) {  // full sort (src/model.c:345-347)
          sort_large(probs, probs2, n, sm);
          token = filter_and_sample(probs, n, p.top_p, p.top_k, rng, sm);
        }
      }
    }
  }

  // the token to every thread, the step, the next embedding; leave the
  // histogram cleared for the next call
  if (threadIdx.x == 0) {
    sm.iwork[4] = token;
    sm.iwork[5] = cs.done == kDoneStopped;
  }
  __syncthreads();
  token = sm.iwork[4];
  if (!sm.iwork[5]) {  // a stopped decode changes nothing
    if (threadIdx.x == 0) finish_step(token, rng, rng_state, io, cs);
    embed_next(token, io);
  }
  if (threadIdx.x < kBuckets) sc.hist[threadIdx.x] = 0;
}

// greedy (src/model.c:143-154): logits untouched, the generator state kept
__global__ __launch_bounds__(1024) void k_sample_greedy(const float* __restrict__ logits, int V,
                                                        uint64_t* __restrict__ rng_state,
                                                        StepIO io) {
  __shared__ Smem sm;
  const CtlSnap cs = ctl_snap(io);
  const int token = argmax_scan(logits, V, -1e9f, sm);
  if (threadIdx.x == 0) sm.iwork[5] = cs.done == kDoneStopped;
  __syncthreads();
  if (sm.iwork[5]) return;  // a stopped decode changes nothing
  if (threadIdx.x == 0) finish_step(token, *rng_state, rng_state, io, cs);
  embed_next(token, io);
}

size_t sample_scratch_bytes(int V) {
  if (V < 1) return 0;
  const size_t lists = (size_t)kFront * front_seg(V);
  // + 32: the two alignments of scratch_of
  return ((size_t)V + lists) * sizeof(Cand) + (2 * kFront + kPBuckets) * sizeof(double) +
         (lists + kPBuckets + 2 * kFront + kBuckets + 1) * sizeof(int) + 32;
}

// pmax/npart: the maxima of logits already scaled by 1/temp (the LM head's
// scaled mode), or nullptr to scale here.  With ctl, the step bookkeeping
// and, with embed, the next embedding row into x[dm]; without, the token to
// out_tokens[0].
hipError_t launch_sample(float* logits, int V, float temp, float min_p, float top_p, int top_k,
                         uint64_t* rng_state, void* scratch, const float* pmax, int npart,
                         int* ctl, int* hist, int* out_tokens, const float* embed, int dm,
                         float* x, hipStream_t s, bool gated) {
  if (V < 1 || V > kMaxVocab) return hipErrorInvalidValue;
  if ((uintptr_t)logits % 16) return hipErrorInvalidValue;  // float4 passes
  const SampleParams p{temp, min_p, top_p, top_k};
  const StepIO io{ctl, hist, out_tokens, embed, dm, x};
  if (temp < 0.05f) {
    hipLaunchKernelGGL(k_sample_greedy, dim3(1), dim3(kThreads), 0, s, logits, V, rng_state, io);
    return hipGetLastError();
  }
  if (!pmax) {
    hipLaunchKernelGGL(k_samp_scale, dim3(kFront), dim3(kFrontThreads), 0, s, logits, V, temp,
                       scratch, gated ? (const int*)ctl : nullptr);
    pmax = scratch_of(scratch, V).pmax;
    npart = kFront;
  }
  const int* gate = gated ? (const int*)ctl : nullptr;
  const dim3 front(kFront), ft(kFrontThreads), one(1), all(kThreads);
  if (effective_k(top_k) > 0) {
    hipLaunchKernelGGL((k_samp_hist<true, false>), front, ft, 0, s, logits, V, p, scratch, pmax,
                       npart, gate);
    hipLaunchKernelGGL((k_sample<true, false>), one, all, 0, s, logits, V, p, rng_state, scratch,
                       pmax, npart, io);
  } else if (tries_parallel(p, V)) {
    hipLaunchKernelGGL((k_samp_hist<false, true>), front, ft, 0, s, logits, V, p, scratch, pmax,
                       npart, gate);
    hipLaunchKernelGGL(k_samp_probs, front, ft, 0, s, V, scratch, gate);
    hipLaunchKernelGGL((k_sample<false, true>), one, all, 0, s, logits, V, p, rng_state, scratch,
                       pmax, npart, io);
  } else {
    hipLaunchKernelGGL((k_samp_hist<false, false>), front, ft, 0, s, logits, V, p, scratch, pmax,
                       npart, gate);
    hipLaunchKernelGGL((k_sample<false, false>), one, all, 0, s, logits, V, p, rng_state, scratch,
                       pmax, npart, io);
  }
  return hipGetLastError();
}

}  // namespace bm

extern "C" size_t bm_hip_sample_workspace_bytes(int vocab) { return bm::sample_scratch_bytes(vocab); }

extern "C" int bm_hip_sample_advanced(float* logits, int vocab, float temp, float min_p,
                                      float top_p, int top_k, uint64_t* rng, void* workspace,
                                      int32_t* token_out, void* stream) {
  if (!logits || !rng || !workspace || !token_out) {
    bm_set_error("sample_advanced: null pointer");
    return -1;
  }
  const hipError_t e =
      bm::launch_sample(logits, vocab, temp, min_p, top_p, top_k, rng, workspace, nullptr, 0,
                        nullptr, nullptr, token_out, nullptr, 0, nullptr, (hipStream_t)stream,
                        false);
  if (e != hipSuccess) {
    bm_set_error("sample_advanced: %s (vocab %d, logits %p; vocab 1..256000, 16-byte aligned logits)",
                 hipGetErrorString(e), vocab, (void*)logits);
    return -1;
  }
  return 0;
}
