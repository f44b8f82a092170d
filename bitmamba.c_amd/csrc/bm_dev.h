// Device helpers shared by the kernel translation units.
#pragma once

#include "bm_common.h"
#include "bm_fp.h"

namespace bm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// 16-byte streaming load (nontemporal: weights are read once per pass)
__device__ __forceinline__ uint4 load_stream16(const void* p) {
  const v4i v = __builtin_nontemporal_load((const v4i*)p);
  return make_uint4((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w);
}

__device__ __forceinline__ uint32_t canon_codes(uint32_t p) {
  // field 11 -> 10: clear the low bit where both bits are set
  return p - (((p >> 1) & p) & 0x55555555u);
}

// ---------------------------------------------------------------------------
// Activation workspace writers
// ---------------------------------------------------------------------------

// 16 int8 values of columns 16g..16g+15 -> split nibbles (unless nib is
// false: the MFMA products read only the permuted bytes) + permuted int8
__device__ __forceinline__ void write_act_group(uint8_t* __restrict__ act_row, int K, int g,
                                                const int (&q)[16], bool nib = true) {
  if (nib) {
  uint32_t le = 0, lo = 0, he = 0, ho = 0;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int xe = q[2 * n], xo = q[2 * n + 1];
    le |= (uint32_t)(xe & 15) << (4 * n);
    lo |= (uint32_t)(xo & 15) << (4 * n);
    he |= (uint32_t)((xe >> 4) & 15) << (4 * n);
    ho |= (uint32_t)((xo >> 4) & 15) << (4 * n);
  }
  *(uint4*)(act_row + act_nib_off(K) + 16 * (size_t)g) = make_uint4(le, lo, he, ho);
  }
  uint32_t pm[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    pm[k] = (uint32_t)(q[k] & 255) | ((uint32_t)(q[4 + k] & 255) << 8) |
            ((uint32_t)(q[8 + k] & 255) << 16) | ((uint32_t)(q[12 + k] & 255) << 24);
  }
  *(uint4*)(act_row + act_perm_off(K) + 16 * (size_t)g) = make_uint4(pm[0], pm[1], pm[2], pm[3]);
}

// Cross-lane reductions on DPP (no LDS round trips).  All 64 lanes must be
// active.  Within a 16-lane row: quad_perm [1,0,3,2] and [2,3,0,1] give
// every lane its quad's value, row_half_mirror pairs the two quads of each
// half row, row_mirror the two half rows.  Rows are then combined through
// scalar reads of lanes 0, 16, 32, 48.
template <int CTRL>
__device__ __forceinline__ int dpp_mov(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}

// sum over the 16 lanes of each row, in every lane of the row
__device__ __forceinline__ int row_sum_i32(int v) {
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0x141>(v);
  v += dpp_mov<0x140>(v);
  return v;
}

__device__ __forceinline__ float row_max_f32(float v) {
  v = fmaxf(v, __int_as_float(dpp_mov<0xB1>(__float_as_int(v))));
  v = fmaxf(v, __int_as_float(dpp_mov<0x4E>(__float_as_int(v))));
  v = fmaxf(v, __int_as_float(dpp_mov<0x141>(__float_as_int(v))));
  v = fmaxf(v, __int_as_float(dpp_mov<0x140>(__float_as_int(v))));
  return v;
}

__device__ __forceinline__ float lane_f32(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// sum / max over the wave, in every lane
__device__ __forceinline__ int wave_sum_i32(int v) {
  v = row_sum_i32(v);
  return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) +
         __builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48);
}

__device__ __forceinline__ float wave_max_f32(float v) {
  v = row_max_f32(v);
  return fmaxf(fmaxf(lane_f32(v, 0), lane_f32(v, 16)), fmaxf(lane_f32(v, 32), lane_f32(v, 48)));
}

// A T-lane row team (T = 16, 32, 64; 16 lanes = one 1024-column slice)
// holding one weight row: reduce each lane's partial x.code over its 16-lane
// slice, subtract the slice's sum of x, and fold the team's slices into the
// fp32 output in slice order (src/kernel.c:255-256, 407-425).
template <int T>
__device__ __forceinline__ float row_finish(int part, int xs_slice, int p_index, int n_slices,
                                            float inv, float o, int unit_base) {
  part = row_sum_i32(part);
  const float f = __fmul_rn((float)(part - xs_slice), inv);
  if constexpr (T == 16) {
    if (p_index < n_slices) o = __fadd_rn(o, f);
  } else {
    // the team's rows (16-lane slices) in order: rows unit_base/16 ..
    const float r[4] = {lane_f32(f, 0), lane_f32(f, 16), lane_f32(f, 32), lane_f32(f, 48)};
#pragma unroll
    for (int q = 0; q < T / 16; ++q) {
      const float fq = T == 64 ? r[q] : (unit_base == 0 ? r[q] : r[2 + q]);
      if (p_index * (T / 16) + q < n_slices) o = __fadd_rn(o, fq);
    }
  }
  return o;
}

// the same team's exact int32 total (x.w over the team's columns)
template <int T>
__device__ __forceinline__ int row_total_i32(int part, int xs_slice, int unit_base) {
  const int t = row_sum_i32(part) - xs_slice;
  if constexpr (T == 16) {
    return t;
  } else {
    const int r[4] = {__builtin_amdgcn_readlane(t, 0), __builtin_amdgcn_readlane(t, 16),
                      __builtin_amdgcn_readlane(t, 32), __builtin_amdgcn_readlane(t, 48)};
    if constexpr (T == 64) return (r[0] + r[1]) + (r[2] + r[3]);
    return unit_base == 0 ? r[0] + r[1] : r[2] + r[3];
  }
}

// ---------------------------------------------------------------------------
// Fast mode (opt-in, not the reference's bits): the sum of squares as one
// balanced pairwise tree over the columns -- 16 consecutive columns per
// leaf group, (((c0+c1)+(c2+c3))+((c4+c5)+(c6+c7)))+..., then the groups
// pairwise in index order -- in place of the four sequential chains.  The
// same tree in every kernel that offers the mode, so a token's prefill and
// decode normalize alike.  (The reduction class of the Metal backend's
// rms_norm_quantize, src/metal/bm_shaders.metal:40-60, not its order.)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float sq_tree16(const float4 (&v)[4]) {
  float t[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    t[k] = __fadd_rn(__fadd_rn(__fmul_rn(v[k].x, v[k].x), __fmul_rn(v[k].y, v[k].y)),
                     __fadd_rn(__fmul_rn(v[k].z, v[k].z), __fmul_rn(v[k].w, v[k].w)));
  return __fadd_rn(__fadd_rn(t[0], t[1]), __fadd_rn(t[2], t[3]));
}

// pairwise over the 16 lanes of each row (every butterfly step adds two
// equal-sized halves, so all lanes of the row hold the same bits), then the
// four rows pairwise: the tree over the wave's 64 leaf groups
__device__ __forceinline__ float wave_tree_f32(float v) {
  v = __fadd_rn(v, __int_as_float(dpp_mov<0xB1>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_mov<0x4E>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_mov<0x141>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_mov<0x140>(__float_as_int(v))));
  return __fadd_rn(__fadd_rn(lane_f32(v, 0), lane_f32(v, 16)),
                   __fadd_rn(lane_f32(v, 32), lane_f32(v, 48)));
}

// the tree's top levels over the G wave sums (1024 columns each)
template <int G>
__device__ __forceinline__ float tree_top(const float* w) {
  if constexpr (G == 1) return w[0];
  if constexpr (G == 2) return __fadd_rn(w[0], w[1]);
  return __fadd_rn(__fadd_rn(w[0], w[1]), __fadd_rn(w[2], w[3]));
}

// ---------------------------------------------------------------------------
// Sum of squares in the four sequential chains (src/kernel.c:77-89), all four
// on one wave
// ---------------------------------------------------------------------------
// chains held in registers (K/64 = E in {16, 32, 64}): lanes 16j..16j+15 of
// the wave own chain j in segments of E consecutive elements; each lane adds
// its segment to the running sum, which then moves one lane up the 16-lane
// row (DPP row_shr:1).  After 16 rounds lane 16j+15 holds chain j's sum.
__host__ __device__ inline int sq_stride_of(int K) { return K / 4 + 68; }

template <int E>
__device__ __forceinline__ float chain_regs(const float* __restrict__ sq, int stride, int lane) {
  const int j = lane >> 4, seg = lane & 15;
  const float* __restrict__ src = sq + j * stride + seg * (E + 4);
  float v[E];
#pragma unroll
  for (int u = 0; u < E / 4; ++u) {
    const float4 t = *(const float4*)(src + 4 * u);
    v[4 * u] = t.x;
    v[4 * u + 1] = t.y;
    v[4 * u + 2] = t.z;
    v[4 * u + 3] = t.w;
  }
  float s = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
#pragma unroll
    for (int k = 0; k < E; ++k) s = __fadd_rn(s, v[k]);
    if (r < 15)
      s = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(s), __float_as_int(s), 0x111,
                                                     0xf, 0xf, false));
  }
  return s;
}

// ---------------------------------------------------------------------------
// The running fp32 sum of a chain of non-negative values (squares), with the
// rounding of every single add kept, by one whole wave instead of one lane.
//
// Lane l holds elements E*l .. E*l+E-1.  While a running sum stays inside one
// binade [2^e, 2^(e+1)), adding c moves its bit pattern by an integer that
// depends on the pattern only through its lowest bit (ties round to even).  So
// each lane runs its E adds twice, from an approximate start p (a prefix sum
// in another order) and from the next float above it.  If both end in p's
// binade and moved by the same integer d, the lane moves every start in the
// binade by d, and the moves of consecutive lanes add up (a prefix sum of
// integers).  The other lanes -- the sum leaves the binade, which happens
// about log2(64) times after lane 0, or a tie makes the two moves differ,
// about as often -- are added up again from their exact start, one after the
// other.  At the end every lane's exact start and end are checked to lie in
// the binade that was assumed for it (the map is monotone, so everything in
// between then does too); if one does not, the chain is added up in turn.
// Infinities and NaNs (exponent 255) are always added up.  Zeros at the end
// leave the sum as it is, so chains are padded with them.
//
// What bounds it: one wave's instruction issue, ~4.7 cycles per dependent add
// (ten lanes added up again cost about as much as everything else).  A chain
// of normal squares takes ~1450 / 2200 cycles at 512 / 1024 elements (K =
// 2048 / 4096), against ~2500 / 5000 for one lane adding in turn; at 256 (K =
// 1024) both take ~1250, and chain_regs stays.  Per launch of the 1B decode:
// out_proj 5.78 -> 4.57 us, in_proj 5.61 -> 5.34; the greedy step, with the
// libm tables in LDS, 0.289 -> 0.265 ms.
// ---------------------------------------------------------------------------
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp_or0(int v) {  // lanes without a source get 0
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}

// inclusive prefix sums over the wave; in fp32 in any order of adds
__device__ __forceinline__ float wave_scan_f32(float v) {
  v = __fadd_rn(v, __int_as_float(dpp_or0<0x111>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_or0<0x112>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_or0<0x114>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_or0<0x118>(__float_as_int(v))));
  v = __fadd_rn(v, __int_as_float(dpp_or0<0x142, 0xa>(__float_as_int(v))));
  return __fadd_rn(v, __int_as_float(dpp_or0<0x143, 0xc>(__float_as_int(v))));
}
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {
  v += (uint32_t)dpp_or0<0x111>((int)v);
  v += (uint32_t)dpp_or0<0x112>((int)v);
  v += (uint32_t)dpp_or0<0x114>((int)v);
  v += (uint32_t)dpp_or0<0x118>((int)v);
  v += (uint32_t)dpp_or0<0x142, 0xa>((int)v);
  return v + (uint32_t)dpp_or0<0x143, 0xc>((int)v);
}

// c: the lane's E elements; start: the sum so far (uniform, >= 0 or NaN);
// returns the sum after all 64 * E elements (uniform).  The first HEAD lanes
// are added up in turn at once, each handing its sum to the next (DPP
// row_shr:1), since the sum doubles often there: worth it for short lanes
// (1B in_proj launch, E = 8: 5.34 us with HEAD = 8, 5.48 with 4, 5.51 with 1;
// out_proj, E = 16: 4.86, 4.77, 4.58).
template <int E>
__device__ __forceinline__ float chain_wave(const float (&c)[E], float start) {
  constexpr uint32_t kBinade = 0x00800000u;  // patterns per binade
  constexpr int HEAD = E <= 8 ? 8 : 1;
  const int lane = threadIdx.x & 63;
  float t[E];
#pragma unroll
  for (int k = 0; k < E; ++k) t[k] = c[k];
#pragma unroll
  for (int w = E / 2; w >= 1; w /= 2)
#pragma unroll
    for (int k = 0; k < w; ++k) t[k] = __fadd_rn(t[k], t[k + w]);
  // the approximate sum before the lane (DPP wave_shr:1 of the prefix sums)
  const float before = __int_as_float(dpp_or0<0x138>(__float_as_int(wave_scan_f32(t[0]))));
  float head = start;
#pragma unroll
  for (int h = 0; h < HEAD; ++h) {
    if (h) head = __int_as_float(dpp_or0<0x111>(__float_as_int(head)));
#pragma unroll
    for (int k = 0; k < E; ++k) head = __fadd_rn(head, c[k]);
  }
  head = lane_f32(head, HEAD - 1);
  const float p = __fadd_rn(head, __fsub_rn(before, lane_f32(before, HEAD)));
  const uint32_t pb = __float_as_uint(p);
  float a = p, b = __uint_as_float(pb + 1);
#pragma unroll
  for (int k = 0; k < E; ++k) {
    a = __fadd_rn(a, c[k]);
    b = __fadd_rn(b, c[k]);
  }
  const uint32_t ab = __float_as_uint(a), bb = __float_as_uint(b);
  const bool moves = (pb ^ bb) < kBinade && pb < 0x7f800000u && bb == ab + 1 && lane >= HEAD;
  const uint32_t d = moves ? ab - pb : 0;
  const uint32_t sum = wave_scan_u32(d);  // moves up to and including the lane

  // the exact sum after a lane is r + sum; r changes at the lanes added up
  // (all lanes add, the one whose turn it is counts)
  uint32_t cur = __float_as_uint(head) + sum, to = cur;
  for (uint64_t left = __ballot(!moves) & (~0ull << HEAD); left;) {
    const int l = __ffsll((unsigned long long)left) - 1;
    left ^= 1ull << l;
    float x = __uint_as_float(cur);
#pragma unroll
    for (int k = 0; k < E; ++k) x = __fadd_rn(x, c[k]);
    cur = (uint32_t)__builtin_amdgcn_readlane((int)(__float_as_uint(x) - sum), l) + sum;
    to = lane >= l ? cur : to;
  }
  const uint32_t from = to - d;
  const bool off = moves && ((to ^ pb) >= kBinade || (from ^ pb) >= kBinade);
  if (__ballot(off) == 0)
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)to, 63));
  // a sum left the binade assumed for its lane: lane by lane
  float x = head;
#pragma unroll 1
  for (int l = HEAD; l < 64; ++l) {
#pragma unroll
    for (int k = 0; k < E; ++k) x = __fadd_rn(x, c[k]);
    x = lane_f32(x, l);
  }
  return x;
}

// LDS layout of a chain for chain_wave: lane l's E elements start at float
// (E + pad) * l, padded by 4 floats where E > 4 so that 16 lanes' 16-byte
// reads fall on different banks
__host__ __device__ constexpr int chain_pad(int E) { return E > 4 ? 4 : 0; }
__host__ __device__ constexpr int chain_floats(int E) { return 64 * (E + chain_pad(E)); }
// elements per lane for chains of K/4 elements, K <= 8192
__host__ __device__ inline int chain_elems(int K) {
  return K <= 1024 ? 4 : (K <= 2048 ? 8 : (K <= 4096 ? 16 : 32));
}

template <int E>
__device__ __forceinline__ float chain_wave_lds(const float* __restrict__ chain, float start) {
  const float* __restrict__ src = chain + (threadIdx.x & 63) * (E + chain_pad(E));
  float c[E];
#pragma unroll
  for (int u = 0; u < E / 4; ++u) {
    const float4 q = *(const float4*)(src + 4 * u);
    c[4 * u] = q.x;
    c[4 * u + 1] = q.y;
    c[4 * u + 2] = q.z;
    c[4 * u + 3] = q.w;
  }
  return chain_wave<E>(c, start);
}

__device__ __forceinline__ float inv_scale_of(float scale_x, float w_scale) {
  return cr_divf(1.0f, __fmul_rn(scale_x, w_scale));  // src/kernel.c:391
}

}  // namespace bm
