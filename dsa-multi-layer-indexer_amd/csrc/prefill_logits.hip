// Indexer scores of many query rows over the same keys (gfx950), the core op
// indexer_logits (attention_core.py:27-49) in the fp8 semantics of the decode
// scan (K:2969-2974, K:2990-2992):
//   logits[b, s, g] = s_k[g] * sum_h w'[b, s, h] * ReLU(q8[b, s, h] . k8[b, g])
// with q and k quantised per 128-element row (quant_core.h) and w' = w * s_q.
//
// The decode scan streams a row's keys past one query; here a thousand query
// rows meet the same keys, so a wave keeps 64 keys in registers (the B operand
// of every product) and the query rows go by through LDS, shared by the
// workgroup's 8 waves.  Per row and 64 keys a wave has 16 MFMAs (512 clocks)
// and 128 VALU operations of ReLU and weight (512 clocks too).  The arithmetic
// is the decode scan's, in its order.
//
// Bound by those two pipes of a SIMD, which overlap only in part (alone 55
// and 57 ns per 4 MFMAs and 32 VALU operations with four waves a SIMD,
// together 81): 1024 rows x 8192 keys x 64 heads in 65 us (2.1
// PFLOP/s of fp8) where the decode scan's flat form took 146 and torch's
// quantisation and page layout 200 before it; here that is 14 (two launches).
// Neither 128 keys a wave, nor the products of the next head group issued
// before this group's sums, nor wave priorities around them moved it by more
// than 3%.
#include <algorithm>

#include "dsa_kernels.h"
#include "quant_core.h"

namespace dsa {

constexpr int kLgThreads = 512;
constexpr int kLgWaves = kLgThreads / kWave;
constexpr int kLgKeys = 64 * kLgWaves;  // 512 keys a workgroup
constexpr int kLgStage = 4;             // query rows staged in LDS at a time

// x [B, T, 128] (DT) -> codes [B, stride, 128] and per-row scale, times w
// when given (wt: its element type); rows past T are zero.  16 lanes a row.
template <int DT>
__global__ __launch_bounds__(256) void quant_rows_kernel(const void* __restrict__ x, long rows, int T, int stride,
                                                         const void* w, int wt, uint8_t* codes, float* scales) {
  const long row = (long)blockIdx.x * 16 + threadIdx.x / 16;
  const int i = threadIdx.x & 15;
  if (row >= rows) return;  // whole 16-lane rows exit together
  const long b = row / stride;
  const int g = (int)(row - b * stride);
  v2u_t c = {0u, 0u};
  float scale = 0.f;
  if (g < T) {
    const long src = b * T + g;
    float v[8];
    load8<DT>(x, src * DSA_INDEX_DIM + 8 * i, v);
    scale = row_scale<true>(v);
    c = quant8<true>(v, scale);
    if (w) scale *= wt == kF32 ? load_elem<kF32>(w, src) : (wt == kBF16 ? load_elem<kBF16>(w, src) : load_elem<kF16>(w, src));
  }
  *reinterpret_cast<v2u_t*>(codes + row * DSA_INDEX_DIM + 8 * i) = c;
  if (i == 0) scales[row] = scale;
}

struct LogitsArgs {
  const uint8_t* q8;   // [B*S, H, 128]
  const float* w;      // [B*S, H]
  const uint8_t* k8;   // [B, Tp, 128], Tp = T rounded up to 64
  const float* ks;     // [B, Tp]
  float* out;          // [B*S, T]
  int B, S, T, ktiles, rows_per_wg, groups;
};

typedef __attribute__((address_space(3))) void* lg_lds_ptr;

template <int NHG>
__global__ __launch_bounds__(kLgThreads, 4) void prefill_logits_kernel(const LogitsArgs A) {
  constexpr int kHeads = 16 * NHG;
  constexpr uint32_t kQBytes = kHeads * DSA_INDEX_DIM;           // one row's queries
  constexpr uint32_t kBufBytes = kLgStage * (kQBytes + kHeads * 4);  // a stage: queries, then weights
  __shared__ __align__(16) uint8_t buf[2 * kBufBytes];
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = wave_id();
  const int kr = lane & 15, kc = lane >> 4;
  const int kt = blockIdx.x % A.ktiles;
  const int grp = (blockIdx.x / A.ktiles) % A.groups, b = blockIdx.x / (A.ktiles * A.groups);
  const int s0 = grp * A.rows_per_wg, s1 = min(A.S, s0 + A.rows_per_wg);
  const int tp = (A.T + 63) / 64 * 64;
  const int g0 = kt * kLgKeys + wv * 64;  // this wave's keys (none when past Tp)

  // ---- the wave's keys: 4 chunks of 16, lane (kr, kc) holds key kr's bytes
  // [32 kc, +32); and key `lane`'s scale ----
  v8i kb[4];
  float ksc = 0.f;
  {
    const bool in = g0 < tp;
    const __amdgpu_buffer_rsrc_t r = dev_rsrc(A.k8 + ((long)b * tp + (in ? g0 : 0)) * DSA_INDEX_DIM, in ? 64 * DSA_INDEX_DIM : 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int off = (16 * j + kr) * DSA_INDEX_DIM + 32 * kc;
      const uint4 x = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
      const uint4 y = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, 0, 0));
      kb[j] = v8i{(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, (int)y.z, (int)y.w};
    }
    if (in) ksc = A.ks[(long)b * tp + g0 + lane];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(kb[j]));  // waited for here
  asm volatile("" : "+v"(ksc));

  // ---- staging: 16-byte chunk c of a stage's queries is chunk c & 7 of head
  // row c >> 3; in LDS its low bits are xored with the head row / 2, so that
  // the 16 heads of an operand read fall in distinct banks.  Direct-to-LDS
  // loads (m0: the wave's base, 16 bytes a lane); rows past the last repeat
  // it. ----
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lg_lds_ptr)buf;
  const uint8_t* qb = A.q8 + (long)b * A.S * kQBytes;
  const float* wb = A.w + (long)b * A.S * kHeads;
  const auto issue = [&](int s, uint32_t at) {
#pragma unroll
    for (int it = 0; it < NHG; ++it) {
      const int c = it * kLgThreads + t;
      const int hrow = c >> 3, j = (c & 7) ^ ((hrow >> 1) & 7);
      const int r = min(s + hrow / kHeads, s1 - 1) - s0;
      const uint32_t off = (uint32_t)r * kQBytes + (uint32_t)(hrow % kHeads) * DSA_INDEX_DIM + 16u * j;
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + at + (uint32_t)(it * kLgThreads + wv * kWave) * 16u);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(dst), "v"(off), "s"(qb + (long)s0 * kQBytes)
                   : "memory", "m0");
    }
    if (wv == 0 && lane < kLgStage * kHeads / 4) {  // the weights, four a lane
      const int r = min(s + lane / (kHeads / 4), s1 - 1) - s0;
      const uint32_t off = (uint32_t)r * kHeads * 4u + (uint32_t)(lane % (kHeads / 4)) * 16u;
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + at + kLgStage * kQBytes);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(dst), "v"(off), "s"(wb + (long)s0 * kHeads)
                   : "memory", "m0");
    }
  };
  // the operand's swizzled chunks 2 kc and 2 kc + 1 of head row kr (the
  // xored bits depend on kr alone)
  const uint32_t qoff0 = (uint32_t)kr * DSA_INDEX_DIM + (uint32_t)((2 * kc) ^ ((kr >> 1) & 7)) * 16u;
  const uint32_t qoff1 = (uint32_t)kr * DSA_INDEX_DIM + (uint32_t)((2 * kc + 1) ^ ((kr >> 1) & 7)) * 16u;
  const auto add32 = [](float x, float y) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  const auto score = [&](int s, const uint8_t* q, const uint8_t* w) {
    float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int hg = 0; hg < NHG; ++hg) {
      const uint4 x = *reinterpret_cast<const uint4*>(q + hg * (16 * DSA_INDEX_DIM) + qoff0);
      const uint4 y = *reinterpret_cast<const uint4*>(q + hg * (16 * DSA_INDEX_DIM) + qoff1);
      const v4f wr = *reinterpret_cast<const v4f*>(w + hg * 64 + kc * 16);
      const v8i qa = v8i{(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, (int)y.z, (int)y.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const v4f z = {0.f, 0.f, 0.f, 0.f};
        const v4f d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(qa, kb[j], z, 0, 0, 0, 0, 0, 0);
        // ReLU on the float's bits (see the decode scan)
#pragma unroll
        for (int r = 0; r < 4; ++r) a[j] += wr[r] * __int_as_float(max(__float_as_int(d[r]), 0));
      }
    }
    const float xs = add32(a[0], a[2]);
    const float ys = add32(a[1], a[3]);
    const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(xs), __float_as_uint(ys), false, false);
    const float acc = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
    // always issued (the wait below counts it); keys past T are outside the
    // resource and dropped
    const __amdgpu_buffer_rsrc_t o = dev_rsrc(A.out + ((long)b * A.S + s) * A.T, (uint32_t)A.T * 4u);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc * ksc), o, 4 * (g0 + lane), 0, 0);
  };

  uint32_t at = 0;
  issue(s0, 0u);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (int s = s0; s < s1; s += kLgStage) {
    __syncthreads();  // this stage has landed (every wave's loads), the other buffer is free
    if (s + kLgStage < s1) issue(s + kLgStage, kBufBytes - at);
    const uint8_t* q = buf + at;
    const uint8_t* w = q + kLgStage * kQBytes;
#pragma unroll
    for (int i = 0; i < kLgStage; ++i)
      if (s + i < s1) score(s + i, q + i * kQBytes, w + i * kHeads * 4);  // uniform
    // the next stage's loads, issued before this stage's 4 stores (every stage
    // but the last is full), have completed; the stores need not have
    static_assert(kLgStage == 4, "the wait below");
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    at = kBufBytes - at;
  }
}

static int logits_tp(int T) { return (T + 63) / 64 * 64; }
static size_t up16(size_t n) { return (n + 15) & ~(size_t)15; }

// [query codes | folded weights | key codes | key scales]
size_t prefill_logits_workspace_bytes(int B, int S, int H, int T) {
  const size_t q = (size_t)B * S * H, k = (size_t)B * logits_tp(T);
  return up16(q * DSA_INDEX_DIM) + up16(q * 4) + up16(k * DSA_INDEX_DIM) + up16(k * 4);
}

static hipError_t launch_quant_rows(const void* x, int dt, int B, int T, int stride, const void* w, int wt,
                                    uint8_t* codes, float* scales, hipStream_t s) {
  const long rows = (long)B * stride;
  const dim3 grid((unsigned)((rows + 15) / 16)), block(256);
  switch (dt) {
    case kF32: hipLaunchKernelGGL(quant_rows_kernel<kF32>, grid, block, 0, s, x, rows, T, stride, w, wt, codes, scales); break;
    case kBF16: hipLaunchKernelGGL(quant_rows_kernel<kBF16>, grid, block, 0, s, x, rows, T, stride, w, wt, codes, scales); break;
    default: hipLaunchKernelGGL(quant_rows_kernel<kF16>, grid, block, 0, s, x, rows, T, stride, w, wt, codes, scales); break;
  }
  return hipGetLastError();
}

hipError_t launch_prefill_logits(const void* q, int qt, const void* k, int kt, const void* w, int wt, void* workspace,
                                 float* out, int B, int S, int H, int T, hipStream_t s) {
  const int tp = logits_tp(T);
  uint8_t* p = static_cast<uint8_t*>(workspace);
  uint8_t* q8 = p;
  p += up16((size_t)B * S * H * DSA_INDEX_DIM);
  float* wq = reinterpret_cast<float*>(p);
  p += up16((size_t)B * S * H * 4);
  uint8_t* k8 = p;
  p += up16((size_t)B * tp * DSA_INDEX_DIM);
  float* ks = reinterpret_cast<float*>(p);
  const int qrows = S * H;
  hipError_t e = launch_quant_rows(q, qt, B, qrows, qrows, w, wt, q8, wq, s);
  if (e == hipSuccess) e = launch_quant_rows(k, kt, B, T, tp, nullptr, 0, k8, ks, s);
  if (e != hipSuccess) return e;
  LogitsArgs A{};
  A.q8 = q8;
  A.w = wq;
  A.k8 = k8;
  A.ks = ks;
  A.out = out;
  A.B = B;
  A.S = S;
  A.T = T;
  A.ktiles = (T + kLgKeys - 1) / kLgKeys;
  // query rows a workgroup: as many workgroups as the chip holds at once (two
  // a CU), in whole stages
  const long per = std::max(1L, 2L * device_cu_count() / std::max(1L, (long)A.ktiles * B));
  A.rows_per_wg = (int)((((long)S + per - 1) / per + kLgStage - 1) / kLgStage * kLgStage);
  A.groups = (S + A.rows_per_wg - 1) / A.rows_per_wg;
  const dim3 grid((unsigned)((long)A.ktiles * A.groups * B)), block(kLgThreads);
  switch (H / 16) {
    case 1: hipLaunchKernelGGL(prefill_logits_kernel<1>, grid, block, 0, s, A); break;
    case 2: hipLaunchKernelGGL(prefill_logits_kernel<2>, grid, block, 0, s, A); break;
    case 3: hipLaunchKernelGGL(prefill_logits_kernel<3>, grid, block, 0, s, A); break;
    default: hipLaunchKernelGGL(prefill_logits_kernel<4>, grid, block, 0, s, A); break;
  }
  return hipGetLastError();
}

}  // namespace dsa
