// Sparse / dense MLA decode of many rows (gfx950): one workgroup takes all the
// keys of a (row, head group).  For calls of the attention alone; in a decode
// layer it stays the decode launch's (decode_main.hip), whose operation it is:
//   out[b,h,:] = sum_j softmax_j(sm * q[b,h,:] . kv_j) * kv_j[:512],
//   kv_j = bf16_rn(f32(e4m3) * scale[d/128]) | bf16 rope.
//
// That kernel's 8 waves share each 128-key tile (gather, QK, softmax, PV, with
// four barriers between them): right for one tile, a chain of waits for
// sixteen.  Here every wave works alone, 16 keys a step: gathered to its
// registers, dequantised, multiplied with the queries (S^T = K Q^T, the key
// rows being the A operand as they were gathered), the probabilities used
// where they come out (O^T = V^T P^T, the MFMA's k order following the
// scores'), the values transposed through a piece of LDS only this wave uses.
// The next 16 rows are in flight from the end of QK on, and the waves' sums
// meet once, at the end.
//
// What bounds it is VALU issue, most of it the dequantisation (2 instructions
// an element, 256 of the ~390 a step).  Two waves a SIMD: with one (4 waves
// of 32 keys) VALU issues at half its rate, and 1024 rows x 2048 keys took
// 321 us; the shared-tile kernel takes 285, this one 230.  Half of the query
// operand stays in registers, the rest is read from LDS: all from LDS 243
// us, more in registers spills.
//
// Each probability enters PV as two bf16 terms, hi + lo, in the two halves of
// a k = 32 MFMA whose A operand repeats the values: 16 keys fill only half of
// that k, and a k = 16 MFMA takes as long.  The result's error against fp64
// (relative norm) is 0.00166, the rounding of the bf16 output alone; with one
// term it was 0.0019-0.0021, as it is in the shared-tile kernel.

#include <type_traits>

#include "dsa_common.h"
#include "dsa_kernels.h"

namespace dsa {

constexpr int kMrWaves = 8;  // two per SIMD
constexpr int kMrThreads = kMrWaves * kWave;
constexpr int kMrKeys = 16;                   // keys a wave's step
constexpr int kMrQLd = DSA_QK_DIM + 8;        // query row stride (bf16): 16 rows on distinct banks
constexpr int kMrQReg = 8;                    // of the 18 query operands, those kept in registers
constexpr int kMrVLd = DSA_LATENT_DIM + 16;   // value row stride (bf16), 8 mod 64 banks
constexpr int kMrOLd = DSA_LATENT_DIM + 4;    // merge row stride (fp32)
constexpr int kMrSlots = kMrWaves / 2;        // waves' sums held at once by the merge
// A wave's sums are relative to its first step's maximum; one that sees a
// score more than 2^32 above it starts over from the true maximum.
constexpr float kMrRise = 32.f;
constexpr size_t kMrQLds = (size_t)kHeadGroup * kMrQLd * 2;
constexpr size_t kMrWaveLds = (size_t)kMrKeys * kMrVLd * 2;
constexpr size_t kMrSlotLds = (size_t)kHeadGroup * kMrOLd * 4;
constexpr size_t kMrLds = kMrWaves * kMrWaveLds + kMrQLds;
static_assert(kMrSlots * kMrSlotLds <= kMrWaves * kMrWaveLds, "the merge's sums fit the value pieces");
static_assert(kMrLds + 2048 <= 160 * 1024, "one CU's LDS");

typedef short v4s_mr __attribute__((ext_vector_type(4)));
typedef v4s_mr __attribute__((address_space(3)))* mr_lds_ptr;

__device__ __forceinline__ v8bf mr_bf8(const uint4& a) {
  v8bf v;
  __builtin_memcpy(&v, &a, 16);
  return v;
}
// op over the four 16-lane groups of a wave, the result in every lane
template <class F>
__device__ __forceinline__ float mr_groups(float v, F op) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(s[0]), __uint_as_float(s[1]));
}

template <bool DENSE>
__global__ __launch_bounds__(kMrThreads, 2) void mla_rows_kernel(const AttnArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ float wm[kMrWaves][kHeadGroup], wl[kMrWaves][kHeadGroup];
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = wave_id();
  const int kr = lane & 15, kc = lane >> 4;
  const int nhg = A.H / kHeadGroup, hg = blockIdx.x % nhg, b = blockIdx.x / nhg;
  const int total = DENSE ? max(0, min(A.dense_lens[b], A.topk)) : A.topk;
  const int steps = (total + kMrKeys - 1) / kMrKeys;
  const int* idx_row = DENSE ? A.dense_pt + (long)b * A.dense_pt_stride : A.idx + (long)b * A.topk;
  const auto slot = [&](int st) {
    const int j = st * kMrKeys + kr;
    if (j >= total) return -1;
    return DENSE ? idx_row[j >> 6] * DSA_PAGE_TOKENS + (j & (DSA_PAGE_TOKENS - 1)) : idx_row[j];
  };

  // the query block, staged once: the B operand (n = head kr), read in the
  // keys' dim order: steps 2i, 2i + 1 -> dims 64i + 16kc + 0..7, + 8..15;
  // 16 + s -> rope dims 32s + 8kc + 0..7
  uint16_t* qs = reinterpret_cast<uint16_t*>(smem + kMrWaves * kMrWaveLds);
  {
    constexpr int kVec = kHeadGroup * DSA_QK_DIM / 8, kRowVec = DSA_QK_DIM / 8;
    const uint4* src = reinterpret_cast<const uint4*>(A.q + ((long)b * A.H + hg * kHeadGroup) * DSA_QK_DIM);
    for (int i = t; i < kVec; i += kMrThreads)
      *reinterpret_cast<uint4*>(qs + (i / kRowVec) * kMrQLd + (i % kRowVec) * 8) = src[i];
  }
  __syncthreads();
  const uint16_t* qrow = qs + kr * kMrQLd;
  const auto q_lds = [&](int s) {
    return *reinterpret_cast<const uint4*>(
        qrow + (s < 16 ? 64 * (s >> 1) + 16 * kc + 8 * (s & 1) : DSA_LATENT_DIM + 32 * (s - 16) + 8 * kc));
  };
  uint4 qreg[kMrQReg];
#pragma unroll
  for (int s = 0; s < kMrQReg; ++s) {
    qreg[s] = q_lds(s);
    asm volatile("" : "+v"(qreg[s].x), "+v"(qreg[s].y), "+v"(qreg[s].z), "+v"(qreg[s].w));  // not read again
  }
  const auto q_op = [&](int s) { return mr_bf8(s < kMrQReg ? qreg[s < kMrQReg ? s : 0] : q_lds(s)); };

  // One step's rows: lane (kr, kc) holds key kr's bytes 64i + 16kc .. + 16 of
  // each 64, the 4 scales, rope bytes 64s + 16kc .. + 16.
  struct Rows {
    uint4 nope[8], rope[2];
    float4 sc;
    bool ok;
  };
  const auto load = [&](int sl, Rows& r) {
    r.ok = sl >= 0 && (long)sl < A.kv_rows;
    const uint8_t* p = A.pool + (long)(r.ok ? sl : 0) * DSA_LATENT_ROW_BYTES;
    const auto read = [&] {
      r.sc = *reinterpret_cast<const float4*>(p + DSA_LATENT_DIM);
#pragma unroll
      for (int i = 0; i < 8; ++i) r.nope[i] = *reinterpret_cast<const uint4*>(p + 64 * i + 16 * kc);
#pragma unroll
      for (int s = 0; s < 2; ++s)
        r.rope[s] = *reinterpret_cast<const uint4*>(p + DSA_LATENT_DIM + 16 + 64 * s + 16 * kc);
    };
    if (__ballot(!r.ok) == 0) {  // uniform: every key is there
      read();
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) r.nope[i] = make_uint4(0, 0, 0, 0);
      r.rope[0] = r.rope[1] = make_uint4(0, 0, 0, 0);
      r.sc = make_float4(0.f, 0.f, 0.f, 0.f);
      if (r.ok) read();
    }
  };

  uint16_t* vt = reinterpret_cast<uint16_t*>(smem + wv * kMrWaveLds);  // [16 keys][dims], this wave's
  const uint16_t* vsrc = vt + (4 * kc + (kr >> 2)) * kMrVLd + 4 * (kr & 3);
  v4f o[32];  // O^T: dims 16 dt + 4 kc + i of head kr
  float m = -INFINITY, l = 0.f;
  bool over = false;

  // r's scores and, unless only their maximum is wanted, its share of the
  // sums; the rows of slots nsl take r's place once QK has read it
  const auto step = [&](auto max_only, Rows& r, int nsl, bool more) {
    constexpr bool kMaxOnly = decltype(max_only)::value;
    asm volatile("" ::: "memory");  // the query operands' reads stay here (hoisted, they spill)
    v4f s = {0.f, 0.f, 0.f, 0.f};
    const float sc4[4] = {r.sc.x, r.sc.y, r.sc.z, r.sc.w};
    uint4* vrow = reinterpret_cast<uint4*>(vt + kr * kMrVLd + 16 * kc);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      uint4 lo, hi;
      dequant16(r.nope[i], sc4[i >> 1], lo, hi);
      s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mr_bf8(lo), q_op(2 * i), s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mr_bf8(hi), q_op(2 * i + 1), s, 0, 0, 0);
      if constexpr (!kMaxOnly) {
        vrow[8 * i] = lo;
        vrow[8 * i + 1] = hi;
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
      s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mr_bf8(r.rope[x]), q_op(16 + x), s, 0, 0, 0);
    // element i is key 4kc + i of head kr; its validity is the gathering
    // lane's (kr = 4kc + i of any group)
    const uint32_t mine = (uint32_t)(__ballot(r.ok) >> (4 * kc));
    if (more) load(nsl, r);
    float tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = mine & (1u << i) ? s[i] * A.sm_log2 : -INFINITY;
      tmax = fmaxf(tmax, s[i]);
    }
    tmax = mr_groups(tmax, [](float x, float y) { return fmaxf(x, y); });
    if constexpr (kMaxOnly) {
      m = fmaxf(m, tmax);
    } else {
      m = m == -INFINITY ? tmax : m;
      over |= tmax > m + kMrRise;
      const float mr = m == -INFINITY ? 0.f : m;
      uint32_t ph[2], pl[2];
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const float p0 = __builtin_amdgcn_exp2f(s[i] - mr), p1 = __builtin_amdgcn_exp2f(s[i + 1] - mr);
        const uint32_t w = pack_bf16x2(p0, p1);
        ph[i >> 1] = w;
        pl[i >> 1] = pack_bf16x2(p0 - __uint_as_float(w << 16), p1 - __uint_as_float(w & 0xffff0000u));
        l += p0 + p1;
      }
      const v8bf pb = mr_bf8(make_uint4(ph[0], ph[1], pl[0], pl[1]));
#pragma unroll
      for (int dt = 0; dt < 32; ++dt) {
        const v2u_t x = __builtin_bit_cast(v2u_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((mr_lds_ptr)(vsrc + 16 * dt)));
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mr_bf8(make_uint4(x[0], x[1], x[0], x[1])), pb, o[dt], 0, 0, 0);
      }
    }
  };
  // this wave's steps wv, wv + 8, ...; the slots one step ahead of the rows
  const auto pass = [&](auto max_only) {
    Rows r;
    int st = wv, sl = slot(st), sl1 = slot(st + kMrWaves);
    if (st < steps) load(sl, r);
    for (; st < steps; st += kMrWaves) {
      const int nx = slot(st + 2 * kMrWaves);
      step(max_only, r, sl1, st + kMrWaves < steps);
      sl1 = nx;
    }
  };
  for (int round = 0;; ++round) {
#pragma unroll
    for (int dt = 0; dt < 32; ++dt) o[dt] = v4f{0.f, 0.f, 0.f, 0.f};
    l = 0.f;
    over = false;
    pass(std::false_type{});
    if (round || __ballot(over) == 0) break;
    m = -INFINITY;
    pass(std::true_type{});
  }

  // the waves' sums meet: wave w takes in wave w + 4's (same lanes, same
  // elements), then the four are added relative to the largest maximum
  l = mr_groups(l, [](float x, float y) { return x + y; });
  if (kc == 0) {
    wm[wv][kr] = m;
    wl[wv][kr] = l;
  }
  __syncthreads();
  float* os = reinterpret_cast<float*>(smem + (wv % kMrSlots) * kMrSlotLds) + kr * kMrOLd + 4 * kc;  // [head][dim]
  if (wv >= kMrSlots)
#pragma unroll
    for (int dt = 0; dt < 32; ++dt) *reinterpret_cast<v4f*>(os + 16 * dt) = o[dt];
  __syncthreads();
  if (wv < kMrSlots) {
    const float m2 = wm[wv + kMrSlots][kr], l2 = wl[wv + kMrSlots][kr];
    const float mm = fmaxf(m, m2);
    const float f1 = m == -INFINITY ? 0.f : exp2f(m - mm), f2 = m2 == -INFINITY ? 0.f : exp2f(m2 - mm);
#pragma unroll
    for (int dt = 0; dt < 32; ++dt) {
      v4f* p = reinterpret_cast<v4f*>(os + 16 * dt);
      *p = o[dt] * f1 + *p * f2;
    }
    if (kc == 0) {
      wm[wv][kr] = mm;
      wl[wv][kr] = l * f1 + l2 * f2;
    }
  }
  __syncthreads();
  const int h = t >> 5, d0 = 4 * (t & 31);
  float mx = -INFINITY, L = 0.f, f[kMrSlots];
#pragma unroll
  for (int w = 0; w < kMrSlots; ++w) mx = fmaxf(mx, wm[w][h]);
#pragma unroll
  for (int w = 0; w < kMrSlots; ++w) {
    f[w] = wm[w][h] == -INFINITY ? 0.f : exp2f(wm[w][h] - mx);
    L += wl[w][h] * f[w];
  }
  const float inv = L > 0.f ? 1.f / L : (L == L ? 0.f : L);  // no key: 0; NaN stays
  uint16_t* out = A.out + ((long)b * A.H + hg * kHeadGroup + h) * DSA_LATENT_DIM + d0;
#pragma unroll
  for (int j = 0; j < DSA_LATENT_DIM / 128; ++j) {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kMrSlots; ++w)
      acc += *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(smem + w * kMrSlotLds) + h * kMrOLd + d0 + 128 * j) * f[w];
    v2u_t w;
    w[0] = pack_bf16x2(acc[0] * inv, acc[1] * inv);
    w[1] = pack_bf16x2(acc[2] * inv, acc[3] * inv);
    *reinterpret_cast<v2u_t*>(out + 128 * j) = w;
  }
}

// Unsplit rows, when there are enough of them to fill the chip (us, 16 heads,
// top-2048, against the shared-tile kernel): 130 rows x 32 heads 100 / 139,
// 300 rows 100 / 139, 1024 rows 230 / 285; 1024 rows of top-512 80 / 108.
// Split rows stay: 100 rows in 2 splits 37 / 40, but 8 splits 21 / 20, with
// a launch more for the merge.  A split count of 1 chosen by a caller with
// fewer rows stays too (its results are compared with riding launches').
bool mla_rows_takes(const AttnArgs& A, int B) { return A.nsplit == 1 && 2 * B * (A.H / kHeadGroup) > device_cu_count(); }

hipError_t launch_mla_rows(const AttnArgs& A, int B, hipStream_t s) {
  static PerDeviceOnce attr;
  const hipError_t e = attr.run([] {
    for (const void* f : {(const void*)mla_rows_kernel<false>, (const void*)mla_rows_kernel<true>})
      if (hipError_t r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMrLds)) return r;
    return hipSuccess;
  });
  if (e != hipSuccess) return e;
  const dim3 grid((unsigned)(B * (A.H / kHeadGroup)));
  if (A.dense_pt) hipLaunchKernelGGL(mla_rows_kernel<true>, grid, dim3(kMrThreads), kMrLds, s, A);
  else hipLaunchKernelGGL(mla_rows_kernel<false>, grid, dim3(kMrThreads), kMrLds, s, A);
  return hipGetLastError();
}

}  // namespace dsa
