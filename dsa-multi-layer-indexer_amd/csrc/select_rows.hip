// Sorted exact top-k of many rows of fp32 scores, one workgroup a row
// (gfx950): the order and rules of dsa_topk with DSA_TOPK_SORTED (reference
// select_topk, attention_core.py:66-91) -- score descending, ties to the
// lower index, NaN above +inf, non-finite selections and missing slots the
// pad value.
//
// A prefill chunk selects for a thousand rows at once, so the chip is filled
// by rows and a row's steps only have to be few:
//   1. load the row into registers (PER keys a thread; PER = 0: a longer row
//      is read again in each step); reduce the finite minimum and maximum;
//   2. count the finite scores in 2048 bins that divide [min, max] evenly by
//      value -- a map that never reverses an order, and that spreads scores
//      over the bins where bits of the key would pile them into a few
//      exponents (and LDS atomics on one address queue up).  The atomic's
//      result is the score's place in its bin;
//   3. a scan from the top bin gives every bin's first output position and
//      the bin T that holds the K-th score;
//   4. scores of bins >= T go to their bin's places in LDS;
//   5. each ranks itself by (key, index) among its bin's few members: its
//      output position.
// So the sort costs a handful of comparisons a score instead of a bitonic
// network's 66 barriers.  A bin of more than kBinMax selected members (many
// equal scores, or a range set by an outlier) takes the general form: t* by
// radix digits, then a bitonic sort.
//
// Bound by the latency of these steps, three rows a CU in flight (78 registers
// for rows of 4097 to 8192 scores: six waves a SIMD).
// 1024 rows of 8192 scores, top-2048: 32 us (1.6 TB/s of scores and int64
// indices), where the slice kernels took 793 (their finalize keeps one row per
// CU: 150 KB of LDS, and sorts it with a barrier a stage); 16384 scores 76, 2048
// scores 16; with every bin crowded (ties) 158.
#include "dsa_common.h"
#include "dsa_kernels.h"

namespace dsa {

constexpr int kSelThreads = 512;
constexpr int kSelWaves = kSelThreads / kWave;
constexpr int kSelBins = 2048;
constexpr int kBinMax = 128;
constexpr int kSelRowMax = 32 * kSelThreads;  // scores held in registers
constexpr int kSelFewRows = 24;               // fewer rows than this,
constexpr int kSelLongRow = 131072;           // longer than this, go to the slice kernels

struct SelShared {
  uint32_t cnt[kSelBins];
  uint32_t off[kSelBins];  // scores in higher bins
  uint32_t tmp[4 * kSelWaves];
  uint32_t res[4];
};

__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float(k & 0x80000000u ? k ^ 0x80000000u : ~k);
}

// exclusive sum over the block in thread order
__device__ __forceinline__ uint32_t sel_scan(uint32_t v, uint32_t* tmp) {
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const uint32_t inc = wave_scan_incl(v);
  if (lane == kWave - 1) tmp[wv] = inc;
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (int w = 0; w < kSelWaves; ++w) before += w < wv ? tmp[w] : 0u;
  __syncthreads();
  return before + inc - v;
}

template <int PER, typename OUT>
__global__ __launch_bounds__(kSelThreads) void select_rows_kernel(const float* __restrict__ scores, const int* lens,
                                                                  int slab, int K, int cap, int pad, OUT* out) {
  extern __shared__ __align__(16) unsigned char smem[];
  SelShared& sh = *reinterpret_cast<SelShared*>(smem);
  uint32_t* ckey = reinterpret_cast<uint32_t*>(smem + sizeof(SelShared));
  uint32_t* cidx = ckey + cap;
  const int t = threadIdx.x;
  const long row = blockIdx.x;
  const int len = lens ? max(0, min(lens[row], slab)) : slab;
  const float* s = scores + row * slab;
  OUT* o = out + row * K;
  const int rounds = PER ? PER : (len + kSelThreads - 1) / kSelThreads;

  // key of position j * 512 + t; 0 (below every real key) past the row
  constexpr int kReg = PER ? PER : 1;
  uint32_t k[kReg], place[kReg];
  if constexpr (PER != 0) {
    float v[kReg];
#pragma unroll
    for (int j = 0; j < kReg; ++j) v[j] = j * kSelThreads + t < len ? s[j * kSelThreads + t] : 0.f;
#pragma unroll
    for (int j = 0; j < kReg; ++j) k[j] = j * kSelThreads + t < len ? rank_key(v[j]) : 0u;
  }
  // f(key, position, register) over this thread's positions; a long row's
  // loads go out in batches
  const auto each = [&](auto&& f) {
    if constexpr (PER != 0) {
#pragma unroll
      for (int j = 0; j < kReg; ++j) f(k[j], j * kSelThreads + t, j);
    } else {
      constexpr int kB = 8;
      for (int j0 = 0; j0 < rounds; j0 += kB) {
        float v[kB];
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int i = (j0 + j) * kSelThreads + t;
          v[j] = i < len ? s[i] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int i = (j0 + j) * kSelThreads + t;
          f(i < len ? rank_key(v[j]) : 0u, i, 0);
        }
      }
    }
  };

  for (int i = t; i < kSelBins; i += kSelThreads) sh.cnt[i] = 0u;
  uint32_t kmin = 0xffffffffu, kmax = 0u, ntop = 0, nfin = 0;
  each([&](uint32_t x, int, int) {
    const bool fin = key_is_finite(x);
    kmin = fin ? min(kmin, x) : kmin;
    kmax = fin ? max(kmax, x) : kmax;
    nfin += fin ? 1u : 0u;
    ntop += x >= kKeyPosInf ? 1u : 0u;
  });
  const uint4 st = block_reduce4<1, 2, 0, 0>(make_uint4(kmin, kmax, ntop, nfin), sh.tmp);
  ntop = st.z;
  // selected finite scores, after the row's NaN and +inf (pads)
  const uint32_t need = st.z >= (uint32_t)K ? 0u : min((uint32_t)K - st.z, st.w);
  for (int i = t; i < K; i += kSelThreads)
    if (i < (int)ntop || i >= (int)(ntop + need)) o[i] = (OUT)pad;
  if (need == 0) return;  // uniform

  float lo = key_value(st.x);
  const float range = key_value(st.y) - lo;
  float scale = (float)(kSelBins - 1) / range;
  // range inf, 0 or denormal: one bin, and lo 0 so that (x - lo) * scale is 0
  // (with an infinite difference it would be NaN, which no integer stands for)
  if (!(range > 0.f) || !(scale > 0.f) || !(scale < INFINITY)) scale = lo = 0.f;
  const auto bin_of = [&](uint32_t x) { return min((int)((key_value(x) - lo) * scale), kSelBins - 1); };
  each([&](uint32_t x, int, int j) {
    if (key_is_finite(x)) {
      const int b = bin_of(x);
      const uint32_t r = atomicAdd(&sh.cnt[b], 1u);
      if constexpr (PER != 0) place[j] = (uint32_t)b | r << 11;
    }
  });
  static_assert(kSelBins == 1 << 11 && kSelRowMax <= 1 << 21, "bin and place share a word");
  __syncthreads();
  // thread t: bins 2047 - 4t .. 2044 - 4t, top down
  {
    static_assert(kSelBins == 4 * kSelThreads, "four bins a thread");
    const int b0 = kSelBins - 4 - 4 * t;
    const uint4 c = *reinterpret_cast<const uint4*>(&sh.cnt[b0]);
    const uint32_t e3 = sel_scan(c.x + c.y + c.z + c.w, sh.tmp);
    const uint32_t e2 = e3 + c.w, e1 = e2 + c.z, e0 = e1 + c.y;
    *reinterpret_cast<uint4*>(&sh.off[b0]) = make_uint4(e0, e1, e2, e3);
    uint32_t big = 0;  // the fullest bin that holds selected scores
    const uint32_t e[4] = {e0, e1, e2, e3}, n[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (e[i] < need) big = max(big, n[i]);
      if (e[i] < need && e[i] + n[i] >= need) sh.res[0] = (uint32_t)(b0 + i);
    }
    big = wave_reduce<2>(big);
    if ((t & (kWave - 1)) == 0) sh.tmp[t / kWave] = big;
  }
  __syncthreads();
  const int T = (int)sh.res[0];
  uint32_t big = 0;
#pragma unroll
  for (int w = 0; w < kSelWaves; ++w) big = max(big, sh.tmp[w]);

  if (big <= (uint32_t)kBinMax) {  // uniform
    const int total = (int)(sh.off[T] + sh.cnt[T]);  // < need + kBinMax <= cap
    if constexpr (PER == 0) {
      __syncthreads();
      for (int i = t; i < kSelBins; i += kSelThreads) sh.cnt[i] = 0u;
      __syncthreads();
    }
    each([&](uint32_t x, int i, int j) {
      if (!key_is_finite(x)) return;
      const int b = PER ? (int)(place[j] & (kSelBins - 1)) : bin_of(x);
      if (b < T) return;
      const uint32_t r = PER ? place[j] >> 11 : atomicAdd(&sh.cnt[b], 1u);
      const uint32_t p = min(sh.off[b] + r, (uint32_t)cap - 1u);  // < cap by construction
      ckey[p] = x;
      cidx[p] = (uint32_t)i;
    });
    __syncthreads();
    for (int p = t; p < total; p += kSelThreads) {
      const uint32_t x = ckey[p], i = cidx[p];
      const int b = bin_of(x);
      const int q0 = (int)sh.off[b], q1 = q0 + (int)sh.cnt[b];
      uint32_t r = (uint32_t)q0;
      for (int q = q0; q < q1; ++q) {
        const uint32_t y = ckey[q];
        r += (y > x || (y == x && cidx[q] < i)) ? 1u : 0u;
      }
      if (r < need) o[ntop + r] = (OUT)i;
    }
    return;
  }

  // ---- a crowded bin: t* among the finite keys by digits 31-21, 20-10, 9-0 ----
  uint32_t prefix = 0, left = need;
  for (int d = 0; d < 3; ++d) {
    const int shift = d == 0 ? 21 : (d == 1 ? 10 : 0), bits = d == 2 ? 10 : 11;
    __syncthreads();
    for (int i = t; i < kSelBins; i += kSelThreads) sh.cnt[i] = 0u;
    __syncthreads();
    each([&](uint32_t x, int, int) {
      if (key_is_finite(x) && (d == 0 || x >> (shift + bits) == prefix))
        atomicAdd(&sh.cnt[(x >> shift) & ((1u << bits) - 1u)], 1u);
    });
    __syncthreads();
    const int b0 = kSelBins - 4 - 4 * t;
    const uint4 c = *reinterpret_cast<const uint4*>(&sh.cnt[b0]);
    const uint32_t e3 = sel_scan(c.x + c.y + c.z + c.w, sh.tmp);
    const uint32_t e2 = e3 + c.w, e1 = e2 + c.z, e0 = e1 + c.y;
    const uint32_t e[4] = {e0, e1, e2, e3}, n[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (e[i] < left && e[i] + n[i] >= left) {
        sh.res[0] = (uint32_t)(b0 + i);
        sh.res[1] = e[i];
      }
    __syncthreads();
    prefix = prefix << bits | sh.res[0];
    left -= sh.res[1];
  }
  const uint32_t tstar = prefix;  // `left` of the keys equal to it are selected, lowest positions first
  if (t == 0) sh.res[2] = 0u;
  uint32_t ties = 0;  // ties seen in earlier rounds (uniform)
  const auto take = [&](uint32_t x, int i) {
    const bool tie = x == tstar;
    uint32_t n;
    const uint32_t before = ties + block_flag_scan(tie, sh.tmp, &n);
    ties += n;
    if (key_is_finite(x) && (x > tstar || (tie && before < left))) {
      const uint32_t p = min(atomicAdd(&sh.res[2], 1u), (uint32_t)cap - 1u);  // < need
      ckey[p] = x;
      cidx[p] = (uint32_t)i;
    }
  };
  __syncthreads();
  if constexpr (PER != 0) {
    each([&](uint32_t x, int i, int) { take(x, i); });
  } else {  // whole rounds of 512 positions, every thread in each (barriers inside)
    for (int j = 0; j < rounds; ++j) {
      const int i = j * kSelThreads + t;
      take(i < len ? rank_key(s[i]) : 0u, i);
    }
  }
  int P = 1;
  while (P < (int)need) P <<= 1;  // <= cap
  for (int i = (int)need + t; i < P; i += kSelThreads) {
    ckey[i] = 0u;
    cidx[i] = 0x7fffffffu;
  }
  for (int w = 2; w <= P; w <<= 1)
    for (int j = w >> 1; j > 0; j >>= 1) {
      __syncthreads();
      for (int i = t; i < P; i += kSelThreads) {
        const int p = i ^ j;
        if (p > i) {
          const uint32_t ka = ckey[i], kb = ckey[p], ia = cidx[i], ib = cidx[p];
          const bool a_first = ka > kb || (ka == kb && ia < ib);
          if (((i & w) == 0) != a_first) {
            ckey[i] = kb;
            ckey[p] = ka;
            cidx[i] = ib;
            cidx[p] = ia;
          }
        }
      }
    }
  __syncthreads();
  for (int i = t; i < (int)need; i += kSelThreads) o[ntop + i] = (OUT)cidx[i];
}

// Everything but a few very long rows, which the slice kernels (topk.hip)
// spread over more workgroups: 1 / 16 / 32 rows of 131072 113 / 115 / 115 us
// here against 111 / 137 / 252, of 200000 163 / 165 / 165 against 114 / 153 /
// 291; 1 / 127 rows of 20000 28 / 30 against 104 / 225.
bool select_rows_takes(int B, int slab, int K) { return K <= 4096 && (slab <= kSelLongRow || B >= kSelFewRows); }

template <int PER, typename OUT>
static hipError_t launch_rows(const float* scores, const int* lens, OUT* out, int B, int slab, int K, int pad,
                              hipStream_t s) {
  int cap = 1;
  while (cap < K) cap <<= 1;
  cap = cap > K + kBinMax ? cap : K + kBinMax;
  const size_t lds = sizeof(SelShared) + 8 * (size_t)cap;
  hipLaunchKernelGGL((select_rows_kernel<PER, OUT>), dim3((unsigned)B), dim3(kSelThreads), lds, s, scores, lens, slab, K,
                     cap, pad, out);
  return hipGetLastError();
}

template <typename OUT>
static hipError_t launch_rows_out(const float* scores, const int* lens, OUT* out, int B, int slab, int K, int pad,
                                  hipStream_t s) {
  if (slab <= 4 * kSelThreads) return launch_rows<4>(scores, lens, out, B, slab, K, pad, s);
  if (slab <= 8 * kSelThreads) return launch_rows<8>(scores, lens, out, B, slab, K, pad, s);
  if (slab <= 16 * kSelThreads) return launch_rows<16>(scores, lens, out, B, slab, K, pad, s);
  if (slab <= kSelRowMax) return launch_rows<32>(scores, lens, out, B, slab, K, pad, s);
  return launch_rows<0>(scores, lens, out, B, slab, K, pad, s);
}

hipError_t launch_select_rows(const float* scores, const int* lens, void* out, int out64, int B, int slab, int K,
                              int pad, hipStream_t s) {
  return out64 ? launch_rows_out(scores, lens, static_cast<int64_t*>(out), B, slab, K, pad, s)
               : launch_rows_out(scores, lens, static_cast<int*>(out), B, slab, K, pad, s);
}

}  // namespace dsa
