// The pieces of xdna::qwen3_stack that are not GEMMs (the GEMMs run on the tile engine's bf16 path),
// for gfx950 (MI355X). The stack runs on a packed activation: the valid tokens of every sequence one
// after another, T rows; the residual stream is float32, GEMM operands bf16 with float32 sums.
//
//   rmsnorm_bf16   y = bf16(w * (x * rsqrt(mean(x^2) + eps)))           Qwen3RMSNorm on float32 rows
//   qk_norm_rope   per token: q / k heads RMSNorm'd over head_dim with their weights, then rotated by
//                  RoPE at the token's position; V written transposed (dims x tokens) for attention
//   attention      softmax(q k^T * scale) v per sequence and head, bidirectional over the sequence's
//                  tokens, grouped-query (q head h reads kv head h / (nh / nkv)), bf16 MFMA with an
//                  online softmax in float32 (32 rows per wave, keys in LDS tiles of 64 or 32)
//   silu_mul       bf16(silu(gate) * up)
//   add_f32        x += y (the residual adds)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "xdna_common.h"
#include "xdna_hip.h"

namespace xdna {

typedef float f32x16s __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8s __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x16s mfma_bf16(const i32x4& a, const i32x4& b, const f32x16s& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8s, a), __builtin_bit_cast(bf16x8s, b), c,
                                                 0, 0, 0);
}

// The sum over the 32 lanes of a half wave, in each of them: neighbours exchanged by DPP (once the lanes of a group
// agree, any lane of the other group will do) and by the row swap, with no trip through the LDS crossbar.
__device__ __forceinline__ float half_wave_sum(float v) {
  auto dpp = [](float x, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value,
                                                                 0xf, 0xf, false));
  };
  v += dpp(v, std::integral_constant<int, 0xb1>{});    // quad_perm 1,0,3,2
  v += dpp(v, std::integral_constant<int, 0x4e>{});    // quad_perm 2,3,0,1
  v += dpp(v, std::integral_constant<int, 0x141>{});   // row_half_mirror
  v += dpp(v, std::integral_constant<int, 0x140>{});   // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float wave_sum(float v) {
  v = half_wave_sum(v);
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int DT>
__device__ __forceinline__ float ld(const void* p, int64_t i) {
  return load_as_f32<DT>(p, i);
}

// Vectors at their elements' alignment (the entry points ask for no more; global loads and stores take them whole).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint16_t u16x4u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32u __attribute__((aligned(2)));

// ------------------------------------------------------------------------------ RMSNorm -> bf16
// W waves per row of d values (d % 256 == 0 and d <= 4096: the host checks), each thread holding up to four groups of
// four consecutive values (thread t: 4 t, then 4 W 64 further on, ...): every load of the row, of the addend and of
// the weight is issued before the first use, so a row costs one round trip to memory and a sum. ADD: the residual
// add that precedes the norm in the layer, x += a, in the same launch (the float32 sums are written back and
// normalized as the separate add and norm would: the same values, one launch fewer). With the add, 1024
// values: 486 rows 2.9 us, 8192 rows 17.8 us (3.7 and 21.3 us with 256 threads of four scalar loads each).
template <int WDT>
__device__ __forceinline__ f32x4 ld4(const void* p, int64_t i) {
  if constexpr (WDT == XDNA_F32) {
    return *reinterpret_cast<const f32x4u*>(static_cast<const float*>(p) + i);
  } else {
    const u16x4u h = *reinterpret_cast<const u16x4u*>(static_cast<const uint16_t*>(p) + i);
    f32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = WDT == XDNA_BF16 ? bf16_bits_to_f32(h[j]) : f16_bits_to_f32(h[j]);
    return r;
  }
}

template <int WDT, bool ADD, int W>
__global__ __launch_bounds__(W * 64) void rmsnorm_bf16_kernel(float* __restrict__ x, const float* __restrict__ a, int d,
                                                              const void* __restrict__ w, float eps,
                                                              uint16_t* __restrict__ y) {
  constexpr int NV = 4;
  __shared__ float red[W];
  const int64_t base = (int64_t)blockIdx.x * d;
  const int i0 = 4 * (int)threadIdx.x;
  f32x4 v[NV], u[NV], g[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = i0 + j * (W * 256);
    const bool in = i < d;                 // d % 256 == 0: a wave is wholly in or out
    v[j] = u[j] = g[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (in) {
      v[j] = *reinterpret_cast<const f32x4u*>(x + base + i);
      if constexpr (ADD) u[j] = *reinterpret_cast<const f32x4u*>(a + base + i);
      g[j] = ld4<WDT>(w, i);
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if constexpr (ADD) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[j][e] = v[j][e] + u[j][e];
      if (i0 + j * (W * 256) < d) *reinterpret_cast<f32x4u*>(x + base + i0 + j * (W * 256)) = v[j];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += v[j][e] * v[j][e];
  }
  ss = wave_sum(ss);
  if constexpr (W > 1) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = red[0];
#pragma unroll
    for (int i = 1; i < W; ++i) ss += red[i];
  }
  const float r = 1.0f / sqrtf(ss / (float)d + eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = i0 + j * (W * 256);
    if (i < d)
      *reinterpret_cast<u32x2u*>(y + base + i) =
          u32x2u{f32x2_to_bf16x2_bits(g[j][0] * (v[j][0] * r), g[j][1] * (v[j][1] * r)),
                 f32x2_to_bf16x2_bits(g[j][2] * (v[j][2] * r), g[j][3] * (v[j][3] * r))};
  }
}

template <int WDT, bool ADD>
int launch_rmsnorm(float* x, const float* a, int64_t rows, int64_t d, const void* w, float eps, uint16_t* y,
                   hipStream_t st) {
  if (d <= 1024) rmsnorm_bf16_kernel<WDT, ADD, 1><<<(unsigned)rows, 64, 0, st>>>(x, a, (int)d, w, eps, y);
  else rmsnorm_bf16_kernel<WDT, ADD, 4><<<(unsigned)rows, 256, 0, st>>>(x, a, (int)d, w, eps, y);
  return launch_status("rmsnorm_bf16");
}

// ------------------------------------------------------------------------------ q / k norm + RoPE
// Two kinds of workgroups. The first V_TOK-token blocks per kv head copy V transposed: 32 tokens x 128 dims come in
// as float2 rows, turn in LDS and leave with 32 tokens side by side in a store instruction (any vt_col; consecutive
// columns make whole 64-byte runs. One dim per lane at one token's column scattered every store over 64 lines).
// The others take one token each: the rotation of its 64 angles once, in LDS, then half a wave per q or k head, lane
// i of it holding dims 2 i, 2 i + 1 and 64 + those, which RoPE rotates into each other (rotate_half), so only the
// norm's sum crosses lanes. 486 tokens 4.0 us, 8192 tokens 30.6 us
// (11.1 and 151.5 us with one wave per (token, head) that computed the angles again and wrote V a value per line).
constexpr int V_TOK = 32;
template <int WDT>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(const float* __restrict__ qkv, int64_t T, int nh, int nkv,
                                                           const void* __restrict__ qw, const void* __restrict__ kw,
                                                           const float* __restrict__ inv_freq,
                                                           const int32_t* __restrict__ pos,
                                                           const int32_t* __restrict__ vt_col, float eps,
                                                           uint16_t* __restrict__ q, uint16_t* __restrict__ k,
                                                           uint16_t* __restrict__ vt, int64_t ld_vt, int64_t vblocks) {
  __shared__ __attribute__((aligned(16))) float buf[V_TOK * 129];
  const int slots = nh + 2 * nkv;
  const int tid = threadIdx.x;
  if ((int64_t)blockIdx.x < vblocks) {
    const int64_t tb = blockIdx.x / nkv;
    const int kvh = (int)(blockIdx.x - tb * nkv);
    const int64_t t0 = tb * V_TOK;
    const int nt = (int)min<int64_t>(V_TOK, T - t0);
    // 129 words a token: 32 tokens of one dim fall on 32 banks
    const float* src = qkv + t0 * slots * 128 + (int64_t)(nh + nkv + kvh) * 128;
    f32x2u v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int tok = min((tid >> 6) + 4 * j, nt - 1);
      v[j] = *reinterpret_cast<const f32x2u*>(src + (int64_t)tok * slots * 128 + 2 * (tid & 63));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int tok = (tid >> 6) + 4 * j;
      buf[tok * 129 + 2 * (tid & 63)] = v[j].x;
      buf[tok * 129 + 2 * (tid & 63) + 1] = v[j].y;
    }
    __syncthreads();
    const int tok = tid & 31;
    if (tok >= nt) return;
    uint16_t* dst = vt + (int64_t)kvh * 128 * ld_vt + vt_col[t0 + tok];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int dim = (tid >> 5) + 8 * j;
      dst[dim * ld_vt] = f32_to_bf16_bits(buf[tok * 129 + dim]);
    }
    return;
  }
  const int64_t t = (int64_t)blockIdx.x - vblocks;
  const int lane = tid & 31, hw = tid >> 5;               // eight half waves
  const float* src = qkv + t * slots * 128;
  float2* const cs = reinterpret_cast<float2*>(buf);      // [64] (cos, sin)
  if (tid < 64) {
    const float f = (float)pos[t] * inv_freq[tid];
    cs[tid] = make_float2(cosf(f), sinf(f));
  }
  __syncthreads();
  const float2 c0 = cs[2 * lane], c1 = cs[2 * lane + 1];
  for (int slot = hw; slot < nh + nkv; slot += 8) {
    const f32x2u a = *reinterpret_cast<const f32x2u*>(src + slot * 128 + 2 * lane);
    const f32x2u b = *reinterpret_cast<const f32x2u*>(src + slot * 128 + 64 + 2 * lane);
    const bool isq = slot < nh;
    const void* w = isq ? qw : kw;
    const float r = 1.0f / sqrtf(half_wave_sum(a.x * a.x + a.y * a.y + b.x * b.x + b.y * b.y) / 128.0f + eps);
    const float ax = ld<WDT>(w, 2 * lane) * (a.x * r), ay = ld<WDT>(w, 2 * lane + 1) * (a.y * r);
    const float bx = ld<WDT>(w, 2 * lane + 64) * (b.x * r), by = ld<WDT>(w, 2 * lane + 65) * (b.y * r);
    uint16_t* dst = (isq ? q + (t * nh + slot) * 128 : k + (t * nkv + (slot - nh)) * 128) + 2 * lane;
    // dim j: x_j cos - x_{j+64} sin; dim j + 64: x_{j+64} cos + x_j sin
    *reinterpret_cast<u32u*>(dst) = f32x2_to_bf16x2_bits(ax * c0.x - bx * c0.y, ay * c1.x - by * c1.y);
    *reinterpret_cast<u32u*>(dst + 64) = f32x2_to_bf16x2_bits(bx * c0.x + ax * c0.y, by * c1.x + ay * c1.y);
  }
}

// ------------------------------------------------------------------------------ attention
// A kv head's queries are its rows: row i of sequence s and kv head g is query i / grp of q head
// g * grp + i % grp (grp = nh / nkv), so the heads that share K and V also share their loads. A workgroup has QW
// waves of 32 rows each and KW groups of such waves; group g takes the key tiles g, g + KW, ... of KT keys, and at
// the end the groups' maxima, sums and outputs meet in LDS. K [KT keys][128] and V^T [128 dims][KT keys] of a tile
// are brought into LDS by the DMA form of the global load. Grid: kv heads fastest, so that with 8 of them each
// XCD's L2 holds the K and V of its own head.
//
// MFMA (srcA = X, srcB = Y) gives, in lane l, row l % 32 of Y and, in element 4 g + r, row 8 g + 4 (l / 32) + r of
// X; lane l supplies values 8 (l / 32) .. + 7 of the 16-deep step of its operand's row l % 32. S = K Q^T: lane l
// <-> row l % 32, elements <-> 16 of 32 keys. O^T = V^T P^T wants keys 8 (l / 32) .. + 7 of each 16-key step in
// lane l; reading K's fragment row i from key swap23(i) (bits 2 and 3 of i exchanged) makes a lane's elements
// 8 u .. 8 u + 7 exactly those of step u, so P goes from one product to the next without leaving its lane.
// LDS chunks of 16 bytes are XORed with the row so that the 16 lanes of a fragment read's phase cover the banks.
//
// Softmax: p = 2^(c (s - m)), c = scale * log2e > 0 (a negative scale goes into Q's sign), in float32; O and l
// are rescaled only in the blocks of 32 keys where some row's running maximum m grows; P is rounded to bf16 for the
// second product, l sums the unrounded p. The maximum follows every 32 keys also where a tile holds 64, and never lags:
// a key that is the maximum has p = 1, which rounds to itself, so the coarser m follows, the further the result is off
// (4096 / 1500 / 700 against 64 bits: 2.237e-3, 2.241e-3 with one maximum per 64 keys, which ran 2 to 10% faster;
// m lagging by up to 2^8: 5% further off and 4% faster; neither is done).
//
// What bounds it: per 64 keys and 32 rows a wave issues 32 MFMAs (1024 cycles of its SIMD) and about 400 vector
// instructions of softmax, so two waves per SIMD (two workgroups per CU, 64 KB of LDS each) fill each other's
// gaps; with the registers for one wave per SIMD only (no spills either way) the long shapes run 1.5x slower.
// Measured, 16 q and 8 kv heads: 1 x 4096 queries 177 us (777 TFLOP/s), 4 x 4096 679 us; lengths 4096 / 1500 / 700
// in one call 215 us against 556 us for one wave per 32 queries of a q head reading its K and V fragments straight
// from memory, 264 / 222 (the split form) 8.7 against 18.7 us. MFMA issue has priority over the other wave's
// softmax (s_setprio): 2% on the long shapes.
__device__ __forceinline__ int swap23(int i) { return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1); }

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef const __attribute__((address_space(1))) void* glb_ptr;
__device__ __forceinline__ void gload_lds16(const void* g, int8_t* l) {   // lane i's 16 bytes land at l + 16 i
  __builtin_amdgcn_global_load_lds((glb_ptr)g, (lds_ptr)l, 16, 0, 0);
}

// the larger of a lane's value and that of lane l ^ 32, and their sum
__device__ __forceinline__ float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __builtin_elementwise_maximum(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// ST: LDS stages of a group. 2: tile t + 1 loads while t is used, one workgroup barrier per tile. 1 (QW == 1, the
// group's LDS is its wave's own, no barriers): the next K loads once S is done, the next V after the tile.
template <int QW, int KW, int KT, int ST>
__global__ __launch_bounds__(QW* KW * 64, 2) void attention_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ vt, int64_t ld_vt,
    const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_len, const int32_t* __restrict__ seq_vt,
    int qblocks, int nh, int nkv, float c, uint32_t qsign, uint16_t* __restrict__ out) {
  static_assert(ST == 2 || QW == 1, "a single stage is one wave's own");
  constexpr int NB = KT / 32;              // 32-key blocks of a tile
  constexpr int KB = KT * 256, VB = KT * 256, STAGE = KB + VB;
  constexpr int NI = KT / 4 / QW;          // 1 KB loads of K, and of V, per wave and tile
  constexpr int VCH = KT / 8, VD = 512 / KT;   // chunks of a V^T row; rows of one 1 KB load
  constexpr int VSH = KT == 64 ? 1 : 2;    // V^T rows per 256 bytes, as a shift
  static_assert(KT == 64 || KT == 32, "V^T rows of 128 or 64 bytes");
  __shared__ __attribute__((aligned(1024))) int8_t lds_all[KW * ST * STAGE];
  __shared__ float ml[KW > 1 ? 2 * KW * 64 : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / QW, qw = wave - kg * QW;
  const int kvh = blockIdx.x % nkv;
  const int sb = blockIdx.x / nkv;
  const int seq = sb / qblocks, qb = sb - seq * qblocks;
  const int n = seq_len[seq];
  const int grp = nh / nkv;
  const int nrows = n * grp;
  if (qb * (QW * 32) >= nrows) return;     // uniform
  const int64_t start = seq_start[seq];
  const int half = lane >> 5, row = lane & 31;
  const int idx = (qb * QW + qw) * 32 + row;
  const int idc = min(idx, nrows - 1);
  const int qi = idc / grp;
  const int64_t qoff = ((start + qi) * nh + (int64_t)kvh * grp + (idc - qi * grp)) * 128;
  i32x4 qf[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    qf[s] = *reinterpret_cast<const i32x4*>(q + qoff + 8 * half + 16 * s);
#pragma unroll
    for (int e = 0; e < 4; ++e) qf[s][e] ^= (int)qsign;
  }
  int8_t* const lds = lds_all + kg * (ST * STAGE);
  const uint16_t* const kbase = k + (start * nkv + kvh) * 128;
  const uint16_t* const vbase = vt + (int64_t)kvh * 128 * ld_vt + seq_vt[seq];
  // this lane's K rows and V^T rows: load j fills 16-byte chunk lane of KB j
  uint32_t krow[NI], kch[NI];
  const uint16_t* vp[NI];
  int vc[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int ld = qw * NI + j;
    krow[j] = (uint32_t)(ld * 4 + (lane >> 4));
    kch[j] = (uint32_t)(((lane & 15) ^ (krow[j] & 15)) * 16);
    const int dim = ld * VD + lane / VCH;
    vc[j] = ((lane & (VCH - 1)) ^ ((dim >> VSH) & (VCH - 1))) * 8;
    vp[j] = vbase + dim * ld_vt + vc[j];
  }
  const uint32_t kpitch = (uint32_t)nkv * 256u;
  // keys past the sequence read its last key (their p are set to 0); V chunks wholly past it read its last chunk
  // (their fragments are set to 0)
  auto load_k = [&](int kb, int8_t* st) {
    const char* base = reinterpret_cast<const char*>(kbase) + (int64_t)kb * kpitch;
    const uint32_t last = (uint32_t)(n - 1 - kb);
#pragma unroll
    for (int j = 0; j < NI; ++j) gload_lds16(base + min(krow[j], last) * kpitch + kch[j], st + ((qw * NI + j) << 10));
  };
  auto load_v = [&](int kb, int8_t* st) {
    if (kb + KT <= n) {
#pragma unroll
      for (int j = 0; j < NI; ++j) gload_lds16(vp[j] + kb, st + KB + ((qw * NI + j) << 10));
    } else {
      const int lastc = (n - 1) & ~7;
#pragma unroll
      for (int j = 0; j < NI; ++j)
        gload_lds16(vp[j] + (min(kb + vc[j], lastc) - vc[j]), st + KB + ((qw * NI + j) << 10));
    }
  };
  f32x16s o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = f32x16s{};
  float m = -INFINITY, l = 0.0f;
  const int krd = swap23(row) * 256;       // the lane's fragment row of each 32-key block
  const int kx = swap23(row) & 15;
  const int vx = (row >> VSH) & (VCH - 1);
  const int nt = (n + KT * KW - 1) / (KT * KW);
  if (kg * KT < n) {
    load_k(kg * KT, lds);
    load_v(kg * KT, lds);
  }
  for (int t = 0; t < nt; ++t) {
    const int kb = (t * KW + kg) * KT;
    const int kn = kb + KW * KT;           // the group's next tile
    int8_t* const cur = lds + (ST == 2 ? (t & 1) * STAGE : 0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    if constexpr (ST == 2) {
      __builtin_amdgcn_s_barrier();        // tile t is whole; every wave is done with tile t - 1
      __builtin_amdgcn_sched_barrier(0);
      if (kn < n) {
        load_k(kn, lds + ((t + 1) & 1) * STAGE);
        load_v(kn, lds + ((t + 1) & 1) * STAGE);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (KW > 1 && kb >= n) continue;       // uniform over the group; the last tile at the earliest
    const bool part = kb + KT > n;         // uniform
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      f32x16s sc = f32x16s{};
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 8; ++s)
        sc = mfma_bf16(*reinterpret_cast<const i32x4*>(cur + b * 8192 + krd + (((2 * s + half) ^ kx) << 4)), qf[s], sc);
      if constexpr (ST == 1) {
        static_assert(ST == 2 || NB == 1, "a single stage holds one block of keys");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (kn < n) load_k(kn, cur);
      }
      __builtin_amdgcn_s_setprio(0);
      float mx = -INFINITY;
      if (part) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (kb + 32 * b + 16 * (e >> 3) + 8 * half + (e & 7) >= n) sc[e] = -INFINITY;
      }
#pragma unroll
      for (int e = 0; e < 16; e += 2)
        mx = __builtin_elementwise_maximum(mx, __builtin_elementwise_maximum(sc[e], sc[e + 1]));
      mx = half_max(mx);
      const bool grow = mx > m;
      if (__builtin_amdgcn_ballot_w64(grow)) {
        const float mn = grow ? mx : m;
        const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * c);
        l *= alpha;
#pragma unroll
        for (int db = 0; db < 4; ++db) o[db] *= alpha;
        m = mn;
      }
      const float mc = m == -INFINITY ? 0.0f : m * c;   // only -inf (or NaN) scores so far: p = 2^-inf = 0, not NaN
      i32x4 pf[2];
      float p[16], ps[2] = {0.0f, 0.0f};
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[e], c, -mc));
        if (part && kb + 32 * b + 16 * (e >> 3) + 8 * half + (e & 7) >= n) p[e] = 0.0f;
      }
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        ps[0] += p[e];
        ps[1] += p[e + 1];
        pf[e >> 3][(e & 7) >> 1] = (int)f32x2_to_bf16x2_bits(p[e], p[e + 1]);
      }
      l += ps[0] + ps[1];
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          i32x4 vf = *reinterpret_cast<const i32x4*>(cur + KB + (db * 32 + row) * (2 * KT) + (((4 * b + 2 * u + half) ^ vx) << 4));
          if (part && kb + 32 * b + 16 * u + 8 * half >= n) vf = i32x4{0, 0, 0, 0};
          o[db] = mfma_bf16(vf, pf[u], o[db]);
        }
      __builtin_amdgcn_s_setprio(0);
    }
    if constexpr (ST == 1) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (kn < n) load_v(kn, cur);
    }
  }
  l = half_sum(l);
  uint16_t* const orow = out + qoff;
  auto store = [&](const f32x16s& v, int db, float inv) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t w0 = f32x2_to_bf16x2_bits(v[4 * g] * inv, v[4 * g + 1] * inv);
      const uint32_t w1 = f32x2_to_bf16x2_bits(v[4 * g + 2] * inv, v[4 * g + 3] * inv);
      *reinterpret_cast<uint2*>(orow + db * 32 + 8 * g + 4 * half) = make_uint2(w0, w1);
    }
  };
  if constexpr (KW == 1) {
    if (idx >= nrows) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int db = 0; db < 4; ++db) store(o[db], db, inv);
  } else {
    // each wave leaves its m, l and O; wave kg then combines dims 32 (4 / KW) kg .. of the 32 rows
    static_assert(QW == 1 && 4 % KW == 0 && KW * 16384 <= KW * ST * STAGE, "one row block, its outputs in LDS");
    __syncthreads();
    ml[kg * 64 + lane] = m;
    ml[(KW + kg) * 64 + lane] = l;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(lds_all + kg * 16384 + (db * 4 + g) * 1024 + lane * 16) =
            f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
    __syncthreads();
    float mt = ml[lane];
#pragma unroll
    for (int g = 1; g < KW; ++g) mt = __builtin_elementwise_maximum(mt, ml[g * 64 + lane]);
    float w[KW], lt = 0.0f;
#pragma unroll
    for (int g = 0; g < KW; ++g) {
      const float mg = ml[g * 64 + lane];
      w[g] = mg == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mg - mt) * c);   // a group without keys: nothing
      lt += ml[(KW + g) * 64 + lane] * w[g];
    }
    if (idx >= nrows) return;              // no barrier follows
    const float inv = 1.0f / lt;
#pragma unroll
    for (int d = 0; d < 4 / KW; ++d) {
      const int db = kg * (4 / KW) + d;
      f32x16s v = f32x16s{};
#pragma unroll
      for (int g = 0; g < KW; ++g)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(lds_all + g * 16384 + (db * 4 + h) * 1024 + lane * 16);
#pragma unroll
          for (int r = 0; r < 4; ++r) v[4 * h + r] += x[r] * w[g];
        }
      store(v, db, inv);
    }
  }
}

// ------------------------------------------------------------------------------ SiLU * up, residual add
__global__ __launch_bounds__(256) void silu_mul_kernel(const float* __restrict__ gu, int64_t T, int64_t inter,
                                                       uint16_t* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= T * inter) return;
  const int64_t t = i / inter, c = i - t * inter;
  const float g = gu[t * 2 * inter + c], u = gu[t * 2 * inter + inter + c];
  y[i] = f32_to_bf16_bits(g / (1.0f + __expf(-g)) * u);
}

__global__ __launch_bounds__(256) void add_f32_kernel(float* __restrict__ x, const float* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] += y[i];
}

}  // namespace xdna

using namespace xdna;

extern "C" {

int xdna_rmsnorm_bf16(const float* x, int64_t rows, int64_t d, const void* w, int w_dtype, float eps, void* y,
                      void* stream) {
  XDNA_REQUIRE(w_dtype == XDNA_F32 || w_dtype == XDNA_BF16 || w_dtype == XDNA_F16, "w_dtype must be F32/BF16/F16");
  XDNA_REQUIRE(rows >= 0 && d >= 256 && d % 256 == 0 && d <= 4096, "d must be a multiple of 256, at most 4096");
  if (rows == 0) return XDNA_OK;
  XDNA_REQUIRE(x && w && y && rows < (1ll << 31), "bad arguments");
  hipStream_t st = as_stream(stream);
  uint16_t* yb = static_cast<uint16_t*>(y);
  float* xm = const_cast<float*>(x);     // read only without ADD
  if (w_dtype == XDNA_F32) return launch_rmsnorm<XDNA_F32, false>(xm, nullptr, rows, d, w, eps, yb, st);
  if (w_dtype == XDNA_BF16) return launch_rmsnorm<XDNA_BF16, false>(xm, nullptr, rows, d, w, eps, yb, st);
  return launch_rmsnorm<XDNA_F16, false>(xm, nullptr, rows, d, w, eps, yb, st);
}

int xdna_add_rmsnorm_bf16(float* x, const float* a, int64_t rows, int64_t d, const void* w, int w_dtype, float eps,
                          void* y, void* stream) {
  XDNA_REQUIRE(w_dtype == XDNA_F32 || w_dtype == XDNA_BF16 || w_dtype == XDNA_F16, "w_dtype must be F32/BF16/F16");
  XDNA_REQUIRE(rows >= 0 && d >= 256 && d % 256 == 0 && d <= 4096, "d must be a multiple of 256, at most 4096");
  if (rows == 0) return XDNA_OK;
  XDNA_REQUIRE(x && a && w && y && rows < (1ll << 31), "bad arguments");
  hipStream_t st = as_stream(stream);
  uint16_t* yb = static_cast<uint16_t*>(y);
  if (w_dtype == XDNA_F32) return launch_rmsnorm<XDNA_F32, true>(x, a, rows, d, w, eps, yb, st);
  if (w_dtype == XDNA_BF16) return launch_rmsnorm<XDNA_BF16, true>(x, a, rows, d, w, eps, yb, st);
  return launch_rmsnorm<XDNA_F16, true>(x, a, rows, d, w, eps, yb, st);
}

int xdna_qk_norm_rope(const float* qkv, int64_t T, int nh, int nkv, const void* q_w, const void* k_w, int w_dtype,
                      const float* inv_freq, const int32_t* pos, const int32_t* vt_col, float eps, void* q, void* k,
                      void* vt, int64_t ld_vt, void* stream) {
  XDNA_REQUIRE(w_dtype == XDNA_F32 || w_dtype == XDNA_BF16 || w_dtype == XDNA_F16, "w_dtype must be F32/BF16/F16");
  XDNA_REQUIRE(T >= 0 && nh >= 1 && nkv >= 1 && nh % nkv == 0, "bad head counts");
  if (T == 0) return XDNA_OK;
  XDNA_REQUIRE(qkv && q_w && k_w && inv_freq && pos && vt_col && q && k && vt && ld_vt >= 1, "bad arguments");
  // tokens of a launch: a workgroup each and nkv per V_TOK of them
  const int64_t most = MAX_LAUNCH_THREADS / 256 / (V_TOK + nkv) * V_TOK;
  XDNA_REQUIRE(most > 0, "too many kv heads");
  hipStream_t st = as_stream(stream);
  for (int64_t t0 = 0; t0 < T; t0 += most) {
    const int64_t n = std::min(most, T - t0), vblocks = cdiv(n, V_TOK) * nkv;
    const dim3 g((unsigned)(vblocks + n));
    const float* x = qkv + t0 * (nh + 2 * (int64_t)nkv) * 128;
    uint16_t *qb = static_cast<uint16_t*>(q) + t0 * nh * 128, *kb = static_cast<uint16_t*>(k) + t0 * nkv * 128,
             *vb = static_cast<uint16_t*>(vt);
#define XDNA_QKR(DT)                                                                                              \
  qk_norm_rope_kernel<DT><<<g, 256, 0, st>>>(x, n, nh, nkv, q_w, k_w, inv_freq, pos + t0, vt_col + t0, eps, qb, kb, vb, \
                                             ld_vt, vblocks)
    if (w_dtype == XDNA_F32) XDNA_QKR(XDNA_F32);
    else if (w_dtype == XDNA_BF16) XDNA_QKR(XDNA_BF16);
    else XDNA_QKR(XDNA_F16);
#undef XDNA_QKR
  }
  return launch_status("qk_norm_rope");
}

int xdna_attention_bf16(const void* q, const void* k, const void* vt, int64_t ld_vt, const int32_t* seq_start,
                        const int32_t* seq_len, const int32_t* seq_vt, int64_t nseq, int64_t max_len, int nh, int nkv,
                        float scale, void* out, void* stream) {
  XDNA_REQUIRE(nseq >= 0 && max_len >= 0 && nh >= 1 && nkv >= 1 && nh % nkv == 0 && nh < 65536, "bad sizes");
  if (nseq == 0 || max_len == 0) return XDNA_OK;
  XDNA_REQUIRE(q && k && vt && seq_start && seq_len && seq_vt && out, "null pointer");
  XDNA_REQUIRE(ld_vt % 8 == 0 && aligned(q, 16) && aligned(k, 16) && aligned(vt, 16) && aligned(out, 8),
               "misaligned operands (ld_vt % 8, 16-byte q / k / vt)");
  const int64_t grp = nh / nkv;
  const float c = fabsf(scale) * 1.44269504088896340736f;
  const uint32_t qsign = scale < 0.0f ? 0x80008000u : 0u;
  // 128 rows per workgroup, sharing each key tile, once such workgroups cover three quarters of the CUs; below that
  // 32 rows with the keys split over four waves, which quarters the chain of tiles a wave walks. Measured, 16 / 8
  // heads, wide against split: one sequence of 512 20.9 / 10.5 us, 1024 36.7 / 22.3, 1300 (168 wide workgroups)
  // 46.6 / 42.2, 1500 (192) 52.2 / 46.6, 1800 62.3 / 61.5, 2048 67.9 / 70.1, 3000 124 / 142; several: eight of 190 (192)
  // 12.0 / 15.7, four of 390 (224) 19.9 / 23.2, four of 500 (256) 22.6 / 26.0. The lengths lie on the GPU, so the
  // workgroups counted are those of nseq sequences of the longest length: 700 / 20 / 20 / 20 takes the wide
  // form, 27.6 / 17.5
  // A wave per 32 keys at the most: sequences of up to 64 take two waves, of up to 32 one, which needs no combination
  // at the end (and no wide form: 64 sequences of 20 6.8 / 7.5 us). One wave / two / four: 20 tokens 4.2 / 4.9 / 5.6 us,
  // 64 tokens 5.2 / 5.0 / 5.7, sixteen of 50 6.8 / 6.6 / 7.9, 97 tokens 7.5 / 6.2 / 5.9
  const bool wide = max_len > 32 && 4 * nseq * cdiv(max_len * grp, 128) * nkv >= 3 * (int64_t)device_cus();
  const int64_t qblocks = cdiv(max_len * grp, wide ? 128 : 32);
  const int64_t threads = wide || max_len > 64 ? 256 : max_len > 32 ? 128 : 64;
  const int64_t step = MAX_LAUNCH_THREADS / threads / (qblocks * nkv);   // sequences per launch
  XDNA_REQUIRE(step > 0, "sequence too long");
  for (int64_t s0 = 0; s0 < nseq; s0 += step) {
    const dim3 g((unsigned)(std::min(step, nseq - s0) * qblocks * nkv));
    const uint16_t *qp = static_cast<const uint16_t*>(q), *kp = static_cast<const uint16_t*>(k),
                   *vp = static_cast<const uint16_t*>(vt);
    uint16_t* op = static_cast<uint16_t*>(out);
#define XDNA_ATT(QW_, KW_, KT_, ST_)                                                                              \
  attention_kernel<QW_, KW_, KT_, ST_><<<g, QW_ * KW_ * 64, 0, as_stream(stream)>>>(                              \
      qp, kp, vp, ld_vt, seq_start + s0, seq_len + s0, seq_vt + s0, (int)qblocks, nh, nkv, c, qsign, op)
    if (wide) XDNA_ATT(4, 1, 64, 2);
    else if (max_len <= 32) XDNA_ATT(1, 1, 32, 1);
    else if (max_len <= 64) XDNA_ATT(1, 2, 32, 1);
    else XDNA_ATT(1, 4, 32, 1);
#undef XDNA_ATT
  }
  return launch_status("attention_bf16");
}

int xdna_silu_mul_bf16(const float* gu, int64_t T, int64_t inter, void* y, void* stream) {
  XDNA_REQUIRE(T >= 0 && inter >= 1, "bad sizes");
  if (T == 0) return XDNA_OK;
  XDNA_REQUIRE(gu && y && cdiv(T * inter, 256) < (1ll << 31), "bad arguments");
  silu_mul_kernel<<<(unsigned)cdiv(T * inter, 256), 256, 0, as_stream(stream)>>>(gu, T, inter,
                                                                                 static_cast<uint16_t*>(y));
  return launch_status("silu_mul_bf16");
}

int xdna_add_f32(float* x, const float* y, int64_t n, void* stream) {
  XDNA_REQUIRE(n >= 0, "bad size");
  if (n == 0) return XDNA_OK;
  XDNA_REQUIRE(x && y && cdiv(n, 256) < (1ll << 31), "bad arguments");
  add_f32_kernel<<<(unsigned)cdiv(n, 256), 256, 0, as_stream(stream)>>>(x, y, n);
  return launch_status("add_f32");
}

}  // extern "C"
