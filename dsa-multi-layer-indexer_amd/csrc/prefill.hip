// Prefill attention on gfx950: many query rows of one request against the
// same keys (reference dense_mla_core, attention_core.py:142-160).
//
//   out[r, :] = sum_j softmax_j(sm * q[r, :] . k_j) * k_j[:512]
//
// over the keys j < limit(r), where row r = (query s, head h) of a request,
// r = s * H + h, sees the first T - S + s + 1 of its T keys.  All heads read
// the same latent keys, so the rows of neighbouring queries are one tall
// matrix against one key block: a contraction on both sides, where the decode
// kernel (16 rows a workgroup) reads and converts every key once per query.
//
// The keys come as bf16 rows of 576: pack_keys_kernel writes, once per call,
// the values that the 656-byte fp8 row format holds (bf16_rn(e4m3 * scale)).
#include <algorithm>

#include "dsa_common.h"
#include "dsa_kernels.h"
#include "quant_core.h"

namespace dsa {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kPfWaves = 4;                 // one per SIMD: the accumulators take half its registers
constexpr int kPfThreads = kPfWaves * kWave;
constexpr int kPfRowsPerWave = 32;
constexpr int kPfRows = kPfWaves * kPfRowsPerWave;  // 128 rows (8 queries of 16 heads) a workgroup
constexpr int kPfKeys = 32;                 // keys a tile
constexpr int kPfDepth = 8;                 // operand fragments read ahead of their MFMA
constexpr int kPfRowChunks = DSA_QK_DIM / 8;        // 72 16-byte chunks of a key row
constexpr int kPfTileBytes = kPfKeys * DSA_QK_DIM * 2;  // 36864
constexpr int kPfLoads = kPfKeys * kPfRowChunks / kPfThreads; // 9 direct-to-LDS loads a thread and tile
static_assert(kPfLoads * kPfThreads == kPfKeys * kPfRowChunks, "whole loads");

constexpr float kPfRise = 32.f;
// A wave takes the second bf16 term of a tile's probabilities too when one of
// its rows has a probability above this share of the row's sum so far; with
// fewer keys a split than kPfBothKeys it always does.
constexpr float kPfSecond = 1.f / 24.f;
constexpr int kPfBothKeys = 512;

struct PrefillArgs {
  const uint16_t* q;     // [B, S*H, 576] bf16
  const uint16_t* keys;  // [B, Tpad, 576] bf16, Tpad = T rounded up to 32
  const uint32_t* mask;  // MASK: [B*S, Tpad / 32], bit j of a query: it attends key j
  uint16_t* out;         // [B, S*H, 512] bf16
  float* part_o;         // nsplit > 1: [nsplit][B*S*H][512]
  float* part_ml;        // [nsplit][B*S*H][2]: (max in log2, sum)
  int B, S, H, T, tiles, nsplit;
  float sm_log2;
};

// LDS position of 16-byte chunk j of key row r: rows are 72 chunks apart (8
// mod 16), so chunk j of 16 consecutive rows would fall on two 16-byte bank
// groups; the low three bits of j are xored with the bit-reversed row / 2,
// which spreads a column over all 16 groups, and a transposed read (8 rows x
// 4 chunks) over 16 as well.
__device__ __forceinline__ int pf_swz(int r) {
  const int x = (r >> 1) & 7;
  return ((x & 1) << 2) | (x & 2) | (x >> 2);
}

__device__ __forceinline__ v4i as_v4i(const uint4& a) { return v4i{(int)a.x, (int)a.y, (int)a.z, (int)a.w}; }
__device__ __forceinline__ v8bf as_bf8(const uint4& a) {
  v8bf v;
  __builtin_memcpy(&v, &a, 16);
  return v;
}

typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef v4s_t __attribute__((address_space(3)))* lds_v4s_ptr;
typedef __attribute__((address_space(1))) const void* gvoid_ptr;
typedef __attribute__((address_space(3))) void* lvoid_ptr;

// max of a value over the two half-waves (lane l and l ^ 32)
__device__ __forceinline__ float half_swap_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_swap_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One workgroup: 128 rows of one request against a range of its keys.
//
// Wave w holds rows [32w, 32w + 32) as the n side of both products: S^T = K
// Q^T (m = 32 keys) leaves a row's scores in one lane pair, so the softmax
// needs one lane swap, and O^T = V^T P^T (m = 32 dims) takes those
// probabilities as its B operand without moving them: the MFMA's k order is
// free, and V's transposed reads follow the order the scores come out in.
// 32 rows a wave halve the LDS bytes a row of 16 would need (8.7 KB a key and
// workgroup, 68 clocks at 128 B each, against 68 clocks of MFMA); their 32 x
// 512 accumulators are the 256 accumulation registers, so the query block
// (144) and the scores live in the 256 vector registers: the QK products are
// written out to say so (the compiler puts every MFMA result in the
// accumulation file and spilled 313), and the accumulators are never
// rescaled (a rescale brought all 256 through the vector file).  Key tiles of
// 32 rows go from memory straight to LDS, two buffers, the next tile in
// flight while this one is used.
//
// Bound by the matrix cores and the LDS reads that feed them: a call with 2999
// causal queries of 16 heads takes 209-220 us by card (156 GFLOP and the second terms of
// the probabilities; a library product of 8192^3 reaches 1218 TFLOP/s here);
// a decode row per query took 1115 us and 2.5 ms of workspace fills.
// Fragments read 4, 6, 8 and 10 steps ahead, with one term: 193, 184, 182 and
// 210 us of kernel.
template <bool MASK, bool BOTH>
__global__ __launch_bounds__(kPfThreads, 1) void prefill_attention_kernel(const PrefillArgs A) {
  __shared__ __align__(16) uint16_t kb[2 * kPfKeys * DSA_QK_DIM];
  __shared__ int redo;
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = wave_id();
  const int n = lane & 31, h = lane >> 5;
  // longest key ranges first: the last row tile sees the most keys
  const int b = blockIdx.x % A.B;
  const int rest = blockIdx.x / A.B;
  const int sp = rest % A.nsplit;
  const int tile = A.tiles - 1 - rest / A.nsplit;
  const int R = A.S * A.H;
  const int r0 = tile * kPfRows;
  const int s_hi = (min(r0 + kPfRows, R) - 1) / A.H;   // last query of the tile
  const int s_lo = r0 / A.H;
  const int kend = A.T - A.S + s_hi + 1;               // keys any row of the tile sees
  const int kfull = A.T - A.S + s_lo + 1;              // keys every row sees
  const int ntile = max(0, (kend + kPfKeys - 1) / kPfKeys);
  const int t0 = (int)((long)ntile * sp / A.nsplit), t1 = (int)((long)ntile * (sp + 1) / A.nsplit);
  const int tpad = (A.T + kPfKeys - 1) / kPfKeys * kPfKeys;
  const uint8_t* kbase = reinterpret_cast<const uint8_t*>(A.keys + (long)b * tpad * DSA_QK_DIM);

  // this lane's row and its limit
  const int row = min(r0 + kPfRowsPerWave * wv + n, R - 1);
  const int limit = A.T - A.S + row / A.H + 1;
  const uint16_t* qrow = A.q + ((long)b * R + row) * DSA_QK_DIM + 8 * h;
  uint4 qf[36];
#pragma unroll
  for (int kk = 0; kk < 36; ++kk) qf[kk] = *reinterpret_cast<const uint4*>(qrow + 16 * kk);
  // waited for here: later the wait would count the key loads in flight too
#pragma unroll
  for (int kk = 0; kk < 36; ++kk) asm volatile("" : : "v"(as_v4i(qf[kk])));

  // source offsets of this thread's loads: LDS chunk p = 256 it + t of the
  // tile holds chunk j of key row p / 72; loads it and it + 9 are 32 rows apart
  uint32_t goff[kPfLoads];
#pragma unroll
  for (int it = 0; it < kPfLoads; ++it) {
    const int p = it * kPfThreads + t;
    const int r = p / kPfRowChunks, jp = p % kPfRowChunks;
    goff[it] = (uint32_t)(r * (DSA_QK_DIM * 2) + ((jp & ~7) | ((jp & 7) ^ pf_swz(r))) * 16);
  }
  // Direct-to-LDS loads, written out because the compiler, which cannot tell
  // the two buffers apart, would wait for them before the next LDS read: the
  // wait is the barrier's (below), one tile later.  m0 holds the wave's LDS
  // base, to which the hardware adds 16 bytes a lane.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lvoid_ptr)kb;
  const auto issue = [&](int tl, uint32_t buf) {
    const uint8_t* src = kbase + (long)tl * kPfTileBytes;
#pragma unroll
    for (int it = 0; it < kPfLoads; ++it) {
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf + (uint32_t)(it * kPfThreads + wv * kWave) * 16u);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(dst), "v"(goff[it]), "s"(src)
                   : "memory", "m0");
    }
  };

  // K operand: row n (+32), chunk 2kk + h
  uint32_t koff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) koff[i] = (uint32_t)(n * (DSA_QK_DIM * 2) + ((2 * i + h) ^ pf_swz(n)) * 16);
  // V operand (transposed read): lane a of a 16-lane group addresses key 4h +
  // (a >> 2) (+8), dims 16 * (group & 1) + 4 (a & 3)
  const int a16 = lane & 15, g1 = (lane >> 4) & 1;
  uint32_t voff[2][2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
#pragma unroll
    for (int e8 = 0; e8 < 2; ++e8) {
      const int r = 4 * h + (a16 >> 2) + 8 * e8;
      const int j = 4 * par + 2 * g1 + ((a16 >> 1) & 1);
      voff[par][e8] = (uint32_t)(r * (DSA_QK_DIM * 2) + (j ^ pf_swz(r)) * 16 + 8 * (a16 & 1));
    }

  v16f o[16];
  float m = -INFINITY, l = 0.f;
  bool over = false;

  const auto compute = [&](auto max_only, int tl, uint32_t bits, const uint16_t* buf) {
    const uint8_t* kp = reinterpret_cast<const uint8_t*>(buf);
    // QK: fragments read kPfDepth steps ahead of their MFMA
    v16f s[2];
    uint4 kf[kPfDepth];
    const auto k_frag = [&](int kk) { return *reinterpret_cast<const uint4*>(kp + koff[kk & 3] + (kk >> 2) * 128); };
#pragma unroll
    for (int i = 0; i < kPfDepth; ++i) kf[i] = k_frag(i);
#pragma unroll
    for (int kk = 0; kk < 36; ++kk) {
      const v4i ka = as_v4i(kf[kk % kPfDepth]), qb = as_v4i(qf[kk]);
      if (kk < 2)
        asm("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[kk]) : "v"(ka), "v"(qb));
      else
        asm("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[kk & 1]) : "v"(ka), "v"(qb));
      if (kk + kPfDepth < 36) kf[kk % kPfDepth] = k_frag(kk + kPfDepth);
    }
    // the matrix unit's results may be read 19 wait states after the last issue
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s[0]), "+v"(s[1]));
#pragma unroll
    for (int e = 0; e < 16; ++e) s[0][e] += s[1][e];
    // scores in the log2 domain; keys at or past the row's limit: -inf.
    // Element i is the tile's key 8 (i / 4) + 4h + (i % 4).
    const int k0 = tl * kPfKeys;
    const bool edge = k0 + kPfKeys > kfull;  // uniform
    float tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float v = s[0][i] * A.sm_log2;
      if constexpr (MASK) v = bits & (1u << (8 * (i >> 2) + (i & 3))) ? v : -INFINITY;
      else if (edge) v = k0 + 8 * (i >> 2) + 4 * h + (i & 3) < limit ? v : -INFINITY;
      s[0][i] = v;
      tmax = fmaxf(tmax, v);
    }
    tmax = half_swap_max(tmax);
    if constexpr (decltype(max_only)::value) {
      m = fmaxf(m, tmax);
      return;
    }
    // The reference point of a row's softmax is its first tile's maximum and
    // stays: any point gives the same result while no probability overflows
    // (bf16 has fp32's exponent range).  A row that rises more than 2^32
    // above it is redone from its true maximum (below): accumulators that
    // are never rescaled stay in the matrix unit's own registers.
    m = m == -INFINITY ? tmax : m;
    over |= tmax > m + kPfRise;
    const float mr = m == -INFINITY ? 0.f : m;
    uint32_t pk[8];
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      s[0][i] = __builtin_amdgcn_exp2f(s[0][i] - mr);
      s[0][i + 1] = __builtin_amdgcn_exp2f(s[0][i + 1] - mr);
      pk[i >> 1] = pack_bf16x2(s[0][i], s[0][i + 1]);
      // the sum of the rounded probabilities, the ones PV multiplies: the
      // weights then add up to one (0-1.3% less error than the unrounded sum)
      l = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, pk[i >> 1]), __builtin_bit_cast(v2bf, 0x3f803f80u),
                                          l, false);
    }
    // PV: 2 steps of 16 keys x 16 blocks of 32 dims, fragments kPfDepth ahead
    const auto v_frag = [&](int i) {
      const int ks = i >> 4, dt = i & 15;
      const uint32_t imm = (dt >> 1) * 128 + ks * (16 * DSA_QK_DIM * 2);
      const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(kp + voff[dt & 1][0] + imm));
      const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr)(kp + voff[dt & 1][1] + imm));
      uint4 vf;
      __builtin_memcpy(&vf.x, &lo, 8);
      __builtin_memcpy(&vf.z, &hi, 8);
      return vf;
    };
    // Probabilities are rounded to bf16, and a row's largest is 1 exactly only
    // when it lies in the row's first tile: with one term the error against
    // 64 bits was up to 4% above that of a softmax about the true maximum.
    // Tiles that hold much of a row's weight take what the rounding left in a
    // second product, which more than makes up for it (kPfSecond):
    // (error, and us a call)        one term      1/16       1/24       1/32     always
    //   2999 queries            0.00200 205  .00177 221  .00173 220  .00171 227  .00162 253
    //   1024 over 2999 keys     0.00195 160  .00190 170  .00186 176  .00183 179  .00166 185
    //   512 over 16384          0.00173 312  .00172 320  .00172 327  .00172 331  .00166 381
    //   1024 over 4096, masked  0.00198 170  .00192 189  .00188 198  .00184 204  .00166 204
    // (a decode row a query, rounded about its running maximum: 0.00196,
    // 0.00192, 0.00172 and 0.00194).
    // what the rounding left of the probabilities, and its sum
    const auto second = [&](uint32_t* w) {
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        w[i >> 1] = pack_bf16x2(s[0][i] - __uint_as_float(pk[i >> 1] << 16),
                                s[0][i + 1] - __uint_as_float(pk[i >> 1] & 0xffff0000u));
        l = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, w[i >> 1]), __builtin_bit_cast(v2bf, 0x3f803f80u),
                                            l, false);
      }
    };
    const auto product = [&](const uint4& v, const uint32_t* p, int i) {
      const uint32_t* pr = p + 4 * (i >> 4);
      o[i & 15] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(v), as_bf8(make_uint4(pr[0], pr[1], pr[2], pr[3])),
                                                          o[i & 15], 0, 0, 0);
    };
    uint4 vf[kPfDepth];
    if constexpr (BOTH) {
      uint32_t pl[8];
      second(pl);
#pragma unroll
      for (int i = 0; i < kPfDepth; ++i) vf[i] = v_frag(i);
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        product(vf[i % kPfDepth], pk, i);
        product(vf[i % kPfDepth], pl, i);
        if (i + kPfDepth < 32) vf[i % kPfDepth] = v_frag(i + kPfDepth);
      }
    } else {
      const bool two = __ballot(__builtin_amdgcn_exp2f(tmax - mr) > kPfSecond * half_swap_sum(l)) != 0;  // uniform
      // one copy of the products in the code: unrolled, or as two branches, the
      // accumulators cross the vector file at the join and spill
#pragma nounroll
      for (int term = 0;; ++term) {
#pragma unroll
        for (int i = 0; i < kPfDepth; ++i) vf[i] = v_frag(i);
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          product(vf[i % kPfDepth], pk, i);
          if (i + kPfDepth < 32) vf[i % kPfDepth] = v_frag(i + kPfDepth);
        }
        if (term || !two) break;
        second(pk);
      }
    }
  };

  const uint32_t* mrow = MASK ? A.mask + ((long)b * A.S + row / A.H) * (tpad / kPfKeys) : nullptr;
  const auto pass = [&](auto max_only) {
    uint32_t cur = 0, bits = 0, next_bits = 0;
    if (t0 < t1) {
      if constexpr (MASK) next_bits = mrow[t0];
      issue(t0, 0u);
    }
    for (int tl = t0; tl < t1; ++tl) {
      if constexpr (MASK) {
        bits = next_bits >> (4 * h);
        asm volatile("" : "+v"(bits));  // waited for here, before the next tile's loads
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // tile tl has landed (every wave's loads), the other buffer is free
      const uint32_t nxt = kPfTileBytes - cur;
      if (tl + 1 < t1) {
        if constexpr (MASK) next_bits = mrow[tl + 1];
        issue(tl + 1, nxt);
      }
      compute(max_only, tl, bits, kb + cur / 2);
      cur = nxt;
    }
    __syncthreads();
  };
  if (t == 0) redo = 0;
  for (int round = 0;; ++round) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[i][e] = 0.f;
    l = 0.f;
    over = false;
    pass(std::false_type{});
    if (round) break;
    if (__ballot(over) && lane == 0) redo = 1;
    __syncthreads();
    if (!redo) break;  // uniform
    m = -INFINITY;
    pass(std::true_type{});
  }

  l = half_swap_sum(l);
  if (r0 + kPfRowsPerWave * wv + n >= R) return;  // rows past the last (no barrier follows)
  // lane (n, h) holds dims 32 dt + 8 (i / 4) + 4h + (i % 4) of its row
  if (A.nsplit == 1) {
    const float inv = l > 0.f ? 1.f / l : (l == l ? 0.f : l);  // a row without a key gives 0, NaN stays
    uint16_t* orow = A.out + ((long)b * R + row) * DSA_LATENT_DIM + 4 * h;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt)
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        v2u_t w;
        w[0] = pack_bf16x2(o[dt][i] * inv, o[dt][i + 1] * inv);
        w[1] = pack_bf16x2(o[dt][i + 2] * inv, o[dt][i + 3] * inv);
        *reinterpret_cast<v2u_t*>(orow + 32 * dt + 2 * i) = w;
      }
  } else {
    const long pr = ((long)sp * A.B + b) * R + row;
    float* po = A.part_o + pr * DSA_LATENT_DIM + 4 * h;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt)
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        v4f w = {o[dt][i], o[dt][i + 1], o[dt][i + 2], o[dt][i + 3]};
        *reinterpret_cast<v4f*>(po + 32 * dt + 2 * i) = w;
      }
    if (h == 0) {
      A.part_ml[2 * pr] = m;
      A.part_ml[2 * pr + 1] = l;
    }
  }
}

// Merge of the key splits of a row: out = sum_s O_s 2^(m_s - m) / sum_s l_s
// 2^(m_s - m), m = max m_s.  One workgroup a row: wave w takes the splits w,
// w + 4, ... (8 dims a lane, 4 splits' loads in flight), then the four sums
// meet in LDS, always in the same order.  Bound by the latency of its loads
// at few rows (64 splits of 16 rows: one wave a row took ~40 us for the
// serial loop), by the partials' bytes at many.
__global__ __launch_bounds__(kPfThreads) void prefill_merge_kernel(const PrefillArgs A) {
  __shared__ float sl[kPfWaves];
  __shared__ v4f so[kPfWaves][2 * kWave];
  const long rows = (long)A.B * A.S * A.H, row = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wv = wave_id();
  float m = -INFINITY;
  for (int s = lane; s < A.nsplit; s += kWave) m = fmaxf(m, A.part_ml[2 * (s * rows + row)]);
  m = wave_max(m);
  const float mr = m == -INFINITY ? 0.f : m;
  float L = 0.f;
  v4f x0 = {0.f, 0.f, 0.f, 0.f}, x1 = x0;
  constexpr int kU = 4;
  for (int s0 = wv; s0 < A.nsplit; s0 += kU * kPfWaves) {
    v4f a[kU], c[kU];
    float ms[kU], ls[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int s = s0 + u * kPfWaves;
      const long pr = (s < A.nsplit ? s : wv) * rows + row;  // past the last: read again, weight 0
      const v4f* po = reinterpret_cast<const v4f*>(A.part_o + pr * DSA_LATENT_DIM) + 2 * lane;
      a[u] = po[0];
      c[u] = po[1];
      ms[u] = A.part_ml[2 * pr];
      ls[u] = A.part_ml[2 * pr + 1];
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (s0 + u * kPfWaves >= A.nsplit) break;  // uniform
      const float w = exp2f(ms[u] - mr);
      L += ls[u] * w;
      x0 += a[u] * w;
      x1 += c[u] * w;
    }
  }
  so[wv][2 * lane] = x0;
  so[wv][2 * lane + 1] = x1;
  if (lane == 0) sl[wv] = L;
  __syncthreads();
  const float tot = (sl[0] + sl[1]) + (sl[2] + sl[3]);
  const float inv = tot > 0.f ? 1.f / tot : (tot == tot ? 0.f : tot);
  if (threadIdx.x < 2 * kWave) {
    const int i = threadIdx.x;
    const v4f o = (so[0][i] + so[1][i]) + (so[2][i] + so[3][i]);
    v2u_t w;
    w[0] = pack_bf16x2(o[0] * inv, o[1] * inv);
    w[1] = pack_bf16x2(o[2] * inv, o[3] * inv);
    *reinterpret_cast<v2u_t*>(A.out + row * DSA_LATENT_DIM + 4 * i) = w;
  }
}

// Key rows [B, T, 576] in fp32 / bf16 / fp16, quantised as the 656-byte row
// format has it: per 128 of the 512 latent dims scale = max(amax, 1e-6) /
// 448, code = e4m3_rne(x / scale); the 64 rope dims bf16_rn.  A NaN or an
// infinity among a group's 128 takes the whole group, as the division by its
// scale does.  ROWS: the 656-byte rows themselves; otherwise the bf16 values
// they hold (bf16_rn(e4m3 * scale), rope), 576 a row.  `stride` output rows a
// request, those past T zero.  One wave a row: lane l holds dims 8l .. 8l + 7,
// a group is 16 lanes, and lanes 0-7 take the rope.
template <int DT, bool ROWS>
__global__ __launch_bounds__(kPfThreads) void pack_keys_kernel(const void* kv, uint8_t* out, int B, int T, int stride) {
  const long row = (long)blockIdx.x * kPfWaves + wave_id();
  if (row >= (long)B * stride) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int b = (int)(row / stride), g = (int)(row % stride);
  uint8_t* dst = out + row * (ROWS ? DSA_LATENT_ROW_BYTES : DSA_QK_DIM * 2);
  if (g >= T) {
    constexpr int kVec = (ROWS ? DSA_LATENT_ROW_BYTES : DSA_QK_DIM * 2) / 16;
    for (int i = lane; i < kVec; i += kWave) reinterpret_cast<uint4*>(dst)[i] = make_uint4(0, 0, 0, 0);
    return;
  }
  const long src = ((long)b * T + g) * DSA_QK_DIM;
  float x[8], r[8];
  load8<DT>(kv, src + 8 * lane, x);
  if (lane < 8) load8<DT>(kv, src + DSA_LATENT_DIM + 8 * lane, r);
  const float scale = row_scale<true>(x);
  const v2u_t code = quant8<true>(x, scale);
  uint32_t rope[4] = {0, 0, 0, 0};
  if (lane < 8)
#pragma unroll
    for (int e = 0; e < 4; ++e) rope[e] = pack_bf16x2(r[2 * e], r[2 * e + 1]);
  if constexpr (ROWS) {
    *reinterpret_cast<v2u_t*>(dst + 8 * lane) = code;
    if ((lane & 15) == 0) *reinterpret_cast<float*>(dst + DSA_LATENT_DIM + (lane >> 2)) = scale;
    if (lane < 8)
      *reinterpret_cast<uint4*>(dst + DSA_LATENT_DIM + 16 + 16 * lane) = make_uint4(rope[0], rope[1], rope[2], rope[3]);
  } else {
    float f[8];
    e4m3x4_to_f32(code[0], f);
    e4m3x4_to_f32(code[1], f + 4);
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = pack_bf16x2(f[2 * e] * scale, f[2 * e + 1] * scale);
    // A tile holds keys that some of its rows do not attend, and 0 * NaN
    // would reach those rows' outputs: a key with a non-finite latent value
    // (its score is NaN whatever the query) keeps a NaN in its rope, which
    // only the scores read, and zeros where the values are read.
    bool bad = false;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      bad |= (w[e] & 0x7f80u) == 0x7f80u || (w[e] & 0x7f800000u) == 0x7f800000u;
    if (__ballot(bad)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = 0u;
      if (lane == 0) rope[0] = 0x7fc07fc0u;
    }
    reinterpret_cast<uint4*>(dst)[lane] = make_uint4(w[0], w[1], w[2], w[3]);
    if (lane < 8) reinterpret_cast<uint4*>(dst)[kWave + lane] = make_uint4(rope[0], rope[1], rope[2], rope[3]);
  }
}

static int prefill_tpad(int T) { return (T + kPfKeys - 1) / kPfKeys * kPfKeys; }

// Selections as sets (reference: the scatter mask, attention_core.py:94-103):
// per query row, idx[0..n) entries outside [0, limit) dropped, repeats
// counted once.  BITS: the row's bitmap of the T keys; otherwise its
// positions ascending, shifted by the batch's first slot, then -1.  One
// workgroup a row over a bitmap in LDS.
constexpr int kSetThreads = 256;
template <typename I, bool BITS>
__global__ __launch_bounds__(kSetThreads) void selection_set_kernel(const I* idx, int n, int S, int T, int words,
                                                                    uint32_t* bits, int* slots) {
  extern __shared__ __align__(16) uint32_t bm[];
  __shared__ uint32_t wsum[kSetThreads / kWave];
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = t / kWave;
  const long row = blockIdx.x;
  const int s = (int)(row % S);
  const int limit = min(T, T - S + s + 1);
  for (int i = t; i < words; i += kSetThreads) bm[i] = 0u;
  __syncthreads();
  const I* src = idx + row * n;
  constexpr int kB = 8;
  for (int i0 = t; i0 < n; i0 += kB * kSetThreads) {
    I v[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) v[j] = i0 + j * kSetThreads < n ? src[i0 + j * kSetThreads] : (I)-1;
#pragma unroll
    for (int j = 0; j < kB; ++j)
      if (v[j] >= 0 && v[j] < (I)limit) atomicOr(&bm[(uint32_t)v[j] >> 5], 1u << ((uint32_t)v[j] & 31u));
  }
  __syncthreads();
  if constexpr (BITS) {
    for (int i = t; i < words; i += kSetThreads) bits[row * words + i] = bm[i];
  } else {
    // thread t: words [t * per, + per); its first output is the count before it
    const int per = (words + kSetThreads - 1) / kSetThreads;
    const int w0 = min(words, t * per), w1 = min(words, w0 + per);
    uint32_t c = 0;
    for (int i = w0; i < w1; ++i) c += (uint32_t)__popc(bm[i]);
    const uint32_t incl = wave_scan_incl<0>(c);
    if (lane == kWave - 1) wsum[wv] = incl;
    __syncthreads();
    uint32_t pos = incl - c, total = 0;
#pragma unroll
    for (int w = 0; w < kSetThreads / kWave; ++w) {
      pos += w < wv ? wsum[w] : 0u;
      total += wsum[w];
    }
    const int base = (int)(row / S) * T;
    int* out = slots + row * n;  // the set has at most n elements
    for (int i = w0; i < w1; ++i)
      for (uint32_t w = bm[i]; w; w &= w - 1u) out[pos++] = base + 32 * i + __builtin_ctz(w);
    for (int i = (int)total + t; i < n; i += kSetThreads) out[i] = -1;
  }
}

// Splits of the keys: with fewer row tiles than CUs, as many as fill the
// chip, each of at least 4 key tiles (a merge pass then follows).
int prefill_nsplit(int B, int S, int H, int T) {
  const long tiles = (long)B * (((long)S * H + kPfRows - 1) / kPfRows);
  const int nkt = prefill_tpad(T) / kPfKeys;
  return (int)std::max(1L, std::min<long>(device_cu_count() / std::max(1L, tiles), nkt / 4));
}

size_t prefill_keys_bytes(int B, int T) { return (size_t)B * prefill_tpad(T) * DSA_QK_DIM * 2; }

size_t prefill_workspace_bytes(int B, int S, int H, int T) {
  const int ns = prefill_nsplit(B, S, H, T);
  return ns == 1 ? 16 : (size_t)ns * B * S * H * (DSA_LATENT_DIM + 2) * sizeof(float);
}

template <bool ROWS>
static hipError_t launch_pack(const void* kv, int dtype, int B, int T, int stride, void* out, hipStream_t s) {
  const dim3 grid((unsigned)(((long)B * stride + kPfWaves - 1) / kPfWaves));
  uint8_t* k = static_cast<uint8_t*>(out);
  switch (dtype) {
    case 0: hipLaunchKernelGGL((pack_keys_kernel<0, ROWS>), grid, dim3(kPfThreads), 0, s, kv, k, B, T, stride); break;
    case 1: hipLaunchKernelGGL((pack_keys_kernel<1, ROWS>), grid, dim3(kPfThreads), 0, s, kv, k, B, T, stride); break;
    default: hipLaunchKernelGGL((pack_keys_kernel<2, ROWS>), grid, dim3(kPfThreads), 0, s, kv, k, B, T, stride); break;
  }
  return hipGetLastError();
}
hipError_t launch_pack_keys(const void* kv, int dtype, int B, int T, void* keys, hipStream_t s) {
  return launch_pack<false>(kv, dtype, B, T, prefill_tpad(T), keys, s);
}
hipError_t launch_pack_rows(const void* kv, int dtype, int B, int T, int stride, void* rows, hipStream_t s) {
  return launch_pack<true>(kv, dtype, B, T, stride, rows, s);
}

int selection_words(int T) { return prefill_tpad(T) / kPfKeys; }

hipError_t launch_selection_set(const void* idx, int idx64, int rows, int n, int S, int T, uint32_t* bits, int* slots,
                                hipStream_t s) {
  const int words = selection_words(T);
  const dim3 grid((unsigned)rows), block(kSetThreads);
  const size_t lds = (size_t)words * 4;
  // the longest context's bitmap and the slots form's sums pass 64 KB together
  static PerDeviceOnce attr;
  const hipError_t e = attr.run([] {
    for (const void* f : {(const void*)selection_set_kernel<int64_t, true>, (const void*)selection_set_kernel<int64_t, false>,
                          (const void*)selection_set_kernel<int, true>, (const void*)selection_set_kernel<int, false>})
      if (hipError_t r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, DSA_SELECTION_MAX_CTX / 8))
        return r;
    return hipSuccess;
  });
  if (e != hipSuccess) return e;
  const auto go = [&](auto kernel, auto* src) {
    hipLaunchKernelGGL(kernel, grid, block, lds, s, src, n, S, T, words, bits, slots);
  };
  if (idx64) {
    const auto* src = static_cast<const int64_t*>(idx);
    if (bits) go(selection_set_kernel<int64_t, true>, src);
    else go(selection_set_kernel<int64_t, false>, src);
  } else {
    const auto* src = static_cast<const int*>(idx);
    if (bits) go(selection_set_kernel<int, true>, src);
    else go(selection_set_kernel<int, false>, src);
  }
  return hipGetLastError();
}

hipError_t launch_prefill_attention(const void* q, const void* keys, const uint32_t* mask, void* workspace, void* out,
                                    int B, int S, int H, int T, float sm_scale, hipStream_t s) {
  PrefillArgs A{};
  A.q = static_cast<const uint16_t*>(q);
  A.keys = static_cast<const uint16_t*>(keys);
  A.mask = mask;
  A.out = static_cast<uint16_t*>(out);
  A.B = B;
  A.S = S;
  A.H = H;
  A.T = T;
  A.tiles = (int)(((long)S * H + kPfRows - 1) / kPfRows);
  A.nsplit = prefill_nsplit(B, S, H, T);
  const long rows = (long)B * S * H;
  A.part_o = static_cast<float*>(workspace);
  A.part_ml = A.part_o + (size_t)A.nsplit * rows * DSA_LATENT_DIM;
  A.sm_log2 = sm_scale * 1.4426950408889634f;
  const dim3 grid((unsigned)((long)A.tiles * A.nsplit * B)), block(kPfThreads);
  // Short key ranges, where most tiles need the second term: always, read
  // once.  (us, always and by need: 300 queries and keys, 75 keys a split,
  // 40.7 and 42.1; 700, 175 keys, 74.1 and 77.2; 1024 over 1200 masked, 344
  // keys, 87.8 and 92.9; 256 over 3000 masked, 32 heads, 718 keys, 103.7 and
  // 105.5; 1500 queries and keys of 32 heads, 750 keys, 189 and 176; 512 over
  // 5000 masked, 1186 keys, 142 and 140; 1024 over 4096 masked, 1792 keys, 205
  // and 192.)
  const bool both = (T - std::min(S, T) / 2) / A.nsplit < kPfBothKeys;
  const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, A); };
  if (mask && both) go(prefill_attention_kernel<true, true>);
  else if (mask) go(prefill_attention_kernel<true, false>);
  else if (both) go(prefill_attention_kernel<false, true>);
  else go(prefill_attention_kernel<false, false>);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && A.nsplit > 1) {
    hipLaunchKernelGGL(prefill_merge_kernel, dim3((unsigned)rows), block, 0, s, A);
    e = hipGetLastError();
  }
  return e;
}

}  // namespace dsa
