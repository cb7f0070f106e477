// Decode-step operand preparation on gfx950: the fp8 quantizers that feed
// the scan and the attention, and the paged appends of one step's keys.
//
// Quantization rule (the reference harness's quantize_e4m3_rowwise,
// K:2969-2974, also the build's fixtures): per 128-element row,
//   scale = max(amax, 1e-6) / 448,  code = e4m3_rne(clamp(x / scale, +-448)),
// with x / scale an IEEE fp32 division and the OCP e4m3fn round to nearest
// even (quant_core.h).
//   - indexer query: one row per (token, head); the scale folds into the
//     head weight, w' = w * scale (K:2984-2985; serving act_quant P:338);
//   - index key: one row per token into the paged cache, 128 codes at slot
//     (g % 64) of page page_table[row, g / 64] and its scale in the page's
//     scale tail (K:540-546, K:2428; serving _store_index_k_cache P:339-342);
//   - latent row: 512 latent values as four 128-element rows (codes + four
//     fp32 scales) and 64 bf16 rope values, packed into the 656-byte row at
//     the token's KV slot (K:1114, K:1355-1395; SGLang's fp8 KV layout).
// Every 128-element row is held by 16 lanes, 8 elements each (16-byte loads,
// 8-byte code stores): a wave takes four query or key rows, or one latent row
// (four groups).  Inputs or caches off those boundaries are read and written
// element by element.
// Bound by memory for a prompt: 8191 tokens x 64 heads (206 MB) in 46 us
// (4.5 TB/s; a large copy 5.0; two or four rows a lane in flight the same); with two elements a lane, a general
// division each and the rounding in integer steps it took 112.
#include "dsa_kernels.h"
#include "quant_core.h"

namespace dsa {

constexpr int kQuantThreads = 256;
constexpr int kQuantRows = kQuantThreads / 16;  // rows a workgroup

template <bool WIDE>
__device__ __forceinline__ void store_codes(uint8_t* dst, v2u_t w) {
  if constexpr (WIDE) {
    *reinterpret_cast<v2u_t*>(dst) = w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) dst[e] = (uint8_t)(w[e >> 2] >> (8 * (e & 3)));
  }
}

// q [rows, 128] bf16 -> codes [rows, 128], w_out[row] = w[row] * scale
template <bool WIDE>
__global__ __launch_bounds__(kQuantThreads) void quant_query_kernel(const void* __restrict__ q, const float* w,
                                                                     uint8_t* codes, float* w_out, long rows) {
  const long row = (long)blockIdx.x * kQuantRows + threadIdx.x / 16;
  const int i = threadIdx.x & 15;
  if (row >= rows) return;  // whole 16-lane rows exit together
  float x[8];
  load8<kBF16, WIDE>(q, row * DSA_INDEX_DIM + 8 * i, x);
  const float scale = row_scale<false>(x);
  store_codes<WIDE>(codes + row * DSA_INDEX_DIM + 8 * i, quant8<false>(x, scale));
  if (i == 0) w_out[row] = w[row] * scale;
}

// keys [n, 128] bf16 of (row[i], pos[i]) -> the paged index cache
template <bool WIDE>
__global__ __launch_bounds__(kQuantThreads) void append_keys_kernel(const void* __restrict__ k, const int* rows,
                                                                     const int* pos, int n, const int* page_table,
                                                                     int pt_stride, uint8_t* pages, long num_pages) {
  const int t = blockIdx.x * kQuantRows + threadIdx.x / 16;
  const int i = threadIdx.x & 15;
  if (t >= n) return;
  const int r = rows[t], g = pos[t];
  const int page = (g >= 0 && g / DSA_PAGE_TOKENS < pt_stride) ? page_table[(long)r * pt_stride + g / DSA_PAGE_TOKENS]
                                                                  : -1;
  float x[8];
  load8<kBF16, WIDE>(k, (long)t * DSA_INDEX_DIM + 8 * i, x);
  const float scale = row_scale<false>(x);
  if (page < 0 || page >= num_pages) return;  // no page for this token: nothing stored
  uint8_t* base = pages + (long)page * DSA_INDEX_PAGE_BYTES;
  const int slot = g % DSA_PAGE_TOKENS;
  store_codes<WIDE>(base + slot * DSA_INDEX_DIM + 8 * i, quant8<false>(x, scale));
  if (i == 0) reinterpret_cast<float*>(base + DSA_PAGE_TOKENS * DSA_INDEX_DIM)[slot] = scale;
}

// latent [n, 576] bf16 -> 656-byte rows at KV slots slot[i], one wave a row:
// 16 lanes a 128-dim group, the 64 rope values copied by lanes 0-31
template <bool WIDE>
__global__ __launch_bounds__(kQuantThreads) void append_latent_kernel(const uint16_t* __restrict__ lat,
                                                                       const int* slots, int n, uint8_t* pool,
                                                                       long kv_rows) {
  const int t = blockIdx.x * (kQuantThreads / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (t >= n) return;
  const long slot = slots[t];
  const uint16_t* src = lat + (long)t * DSA_QK_DIM;
  float x[8];
  load8<kBF16, WIDE>(src, 8 * lane, x);
  const float scale = row_scale<false>(x);
  if (slot < 0 || slot >= kv_rows) return;
  uint8_t* dst = pool + slot * DSA_LATENT_ROW_BYTES;
  store_codes<WIDE>(dst + 8 * lane, quant8<false>(x, scale));
  if ((lane & 15) == 0) reinterpret_cast<float*>(dst + DSA_LATENT_DIM)[lane >> 4] = scale;
  if (lane < 32) {
    uint16_t* rope = reinterpret_cast<uint16_t*>(dst + DSA_LATENT_DIM + 16);
    if constexpr (WIDE) {
      reinterpret_cast<uint32_t*>(rope)[lane] = reinterpret_cast<const uint32_t*>(src + DSA_LATENT_DIM)[lane];
    } else {
      rope[2 * lane] = src[DSA_LATENT_DIM + 2 * lane];
      rope[2 * lane + 1] = src[DSA_LATENT_DIM + 2 * lane + 1];
    }
  }
}

static bool wide_ok(const void* in, const void* out) { return ((uintptr_t)in & 15) == 0 && ((uintptr_t)out & 7) == 0; }

hipError_t launch_quant_query(const void* q_bf16, const float* w, void* codes, float* w_out, long rows,
                              hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  const dim3 grid((unsigned)((rows + kQuantRows - 1) / kQuantRows));
  uint8_t* c = static_cast<uint8_t*>(codes);
  if (wide_ok(q_bf16, codes))
    hipLaunchKernelGGL(quant_query_kernel<true>, grid, dim3(kQuantThreads), 0, s, q_bf16, w, c, w_out, rows);
  else
    hipLaunchKernelGGL(quant_query_kernel<false>, grid, dim3(kQuantThreads), 0, s, q_bf16, w, c, w_out, rows);
  return hipGetLastError();
}

hipError_t launch_append_keys(const void* k_bf16, const int* rows, const int* pos, int n, const int* page_table,
                              int pt_stride, void* pages, long num_pages, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const dim3 grid((unsigned)((n + kQuantRows - 1) / kQuantRows));
  uint8_t* p = static_cast<uint8_t*>(pages);
  if (wide_ok(k_bf16, pages))
    hipLaunchKernelGGL(append_keys_kernel<true>, grid, dim3(kQuantThreads), 0, s, k_bf16, rows, pos, n, page_table,
                       pt_stride, p, num_pages);
  else
    hipLaunchKernelGGL(append_keys_kernel<false>, grid, dim3(kQuantThreads), 0, s, k_bf16, rows, pos, n, page_table,
                       pt_stride, p, num_pages);
  return hipGetLastError();
}

hipError_t launch_append_latent(const void* lat_bf16, const int* slots, int n, void* pool, long kv_rows,
                                hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const dim3 grid((unsigned)((n + kQuantThreads / kWave - 1) / (kQuantThreads / kWave)));
  const uint16_t* lat = static_cast<const uint16_t*>(lat_bf16);
  uint8_t* p = static_cast<uint8_t*>(pool);
  if (wide_ok(lat_bf16, pool))
    hipLaunchKernelGGL(append_latent_kernel<true>, grid, dim3(kQuantThreads), 0, s, lat, slots, n, p, kv_rows);
  else
    hipLaunchKernelGGL(append_latent_kernel<false>, grid, dim3(kQuantThreads), 0, s, lat, slots, n, p, kv_rows);
  return hipGetLastError();
}

}  // namespace dsa
