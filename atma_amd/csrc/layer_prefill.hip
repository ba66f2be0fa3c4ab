// Small launches around the global layer's prefill, each one for a chain of eager ops whose launches cost more than their
// work (a short prompt's layer is bound by them: 2,999 tokens spend about 0.4 ms in kernels and took 0.8 ms):
//
//  * memory_gate_logits: the memory branch's two gate projections (model/blocks.py:466-467, H outputs each) in fp32
//    from one pass over the rows, where two GEMMs of 8 columns read the rows twice and round to 16 bits.  Bound by the
//    rows' read: a workgroup is 16 rows x up to 32 outputs on v_mfma_f32_16x16x32, its four waves splitting K so that
//    every load of a short prompt is in flight at once, the waves' sums meeting in LDS in a fixed order (deterministic).
//  * polar_params_f32: the five Polar parameter tensors widened to fp32 into one buffer.
//  * paged_kv_concat: a sequence's cached K / V rows gathered from its pages, then a chunk's rows, into contiguous rows
//    (inference/models/atma.py:509-544 gathers the pages and concatenates, four copies).
#include "common.h"

namespace atma {

struct GateLogitArgs {
  const void* x;  // (M, K) rows
  int64_t ldx;
  const void* w[2];  // (H, K) contiguous
  const void* bias[2];  // (H,) or null
  float* out[2];        // (M, H)
  int64_t M;
  int K, H;
};

template <typename T, int NT>
__global__ void __launch_bounds__(256) gate_logits_kernel(GateLogitArgs a) {
  __shared__ f32x4 part[4][NT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * 16;
  const int kw = a.K / 4;  // a wave's share, a multiple of 32
  const T* x = (const T*)a.x + min(m0 + r, a.M - 1) * a.ldx + wave * kw + 8 * g;
  const T* w[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = min(16 * t + r, 2 * a.H - 1);  // columns past 2 H repeat the last and are dropped
    w[t] = (const T*)a.w[n >= a.H] + (int64_t)(n >= a.H ? n - a.H : n) * a.K + wave * kw + 8 * g;
  }
  f32x4 acc[NT] = {};
#pragma unroll 8
  for (int k = 0; k < kw; k += 32) {
    const u32x4 xv = *(const u32x4*)(x + k);
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = mfma16x16x32<T>(xv, *(const u32x4*)(w[t] + k), acc[t]);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) part[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= NT) return;
  f32x4 s = part[0][wave][lane];
#pragma unroll
  for (int q = 1; q < 4; ++q) s += part[q][wave][lane];
  const int n = 16 * wave + r;
  if (n >= 2 * a.H) return;
  const int which = n >= a.H, h = n - which * a.H;
  const float b = a.bias[which] ? to_f32(((const T*)a.bias[which])[h]) : 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + 4 * g + i;
    if (m < a.M) a.out[which][m * a.H + h] = s[i] + b;
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
params_f32_kernel(const T* v_null, const T* p0, const T* p1, const T* p2, const T* p3, float* out, int H, int Hd) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < Hd) {
    out[i] = to_f32(v_null[i]);
  } else if (i < Hd + 4 * H) {
    const int j = i - Hd, which = j / H, h = j - which * H;
    const T* p = which == 0 ? p0 : which == 1 ? p1 : which == 2 ? p2 : p3;
    out[i] = to_f32(p[h]);
  }
}

struct ConcatArgs {
  const u32x4 *cache[2], *tail[2];  // pages of rows; the chunk's rows
  u32x4* out[2];
  const int32_t* pages;
  int64_t cached, rows;  // rows from the pages; rows in all
  int64_t tail_st[2];    // 16-byte vectors between the chunk's rows
  int64_t num_pages;
  int page, vecs;  // rows of a page; 16-byte vectors of a row
};

// Four vectors a thread, every load issued before the first store.
__global__ void __launch_bounds__(256) kv_concat_kernel(ConcatArgs a) {
  const int which = blockIdx.y;
  const int64_t n = a.rows * a.vecs, stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  u32x4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t j = i + u * stride;
    v[u] = u32x4{0u, 0u, 0u, 0u};
    if (j < n) {
      const int64_t row = j / a.vecs, e = j - row * a.vecs;
      if (row < a.cached) {
        const int64_t pg = a.pages[row / a.page];
        if (pg >= 0 && pg < a.num_pages) v[u] = a.cache[which][(pg * a.page + row % a.page) * a.vecs + e];
      } else {
        v[u] = a.tail[which][(row - a.cached) * a.tail_st[which] + e];
      }
    }
  }
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (i + u * stride < n) a.out[which][i + u * stride] = v[u];
}

static bool lp_al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

template <typename T>
static int launch_gate_logits(const GateLogitArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.M + 15) / 16));
  if (a.H <= 8) gate_logits_kernel<T, 1><<<grid, dim3(256), 0, s>>>(a);
  else gate_logits_kernel<T, 2><<<grid, dim3(256), 0, s>>>(a);
  return check_launch("memory_gate_logits");
}

template <typename T>
static int launch_params(const void* const* p, float* out, int64_t H, int64_t d, hipStream_t s) {
  const int Hd = (int)(H * d), n = Hd + 4 * (int)H;
  params_f32_kernel<T><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(
      (const T*)p[0], (const T*)p[1], (const T*)p[2], (const T*)p[3], (const T*)p[4], out, (int)H, Hd);
  return check_launch("polar_params_f32");
}

}  // namespace atma

using namespace atma;

extern "C" int atma_memory_gate_logits(const void* x, int64_t ldx, const void* wg, const void* bg, const void* wb,
                                       const void* bb, float* zg, float* zb, int64_t M, int64_t K, int64_t H, int dtype,
                                       void* stream) {
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "memory_gate_logits: 16-bit rows only (dtype %d)", dtype);
  if (H < 1 || H > 16 || K < 128 || K % 128 || K > 1 << 20)
    return set_error(ATMA_ERR_UNSUPPORTED, "memory_gate_logits: 1 to 16 heads, K a multiple of 128");
  if (M < 0 || M > 0x7fffffff) return set_error(ATMA_ERR_INVALID, "memory_gate_logits: bad sizes");
  if (M == 0) return ATMA_OK;
  if (!x || !wg || !wb || !zg || !zb) return set_error(ATMA_ERR_INVALID, "memory_gate_logits: null pointer");
  if (!lp_al16(x) || !lp_al16(wg) || !lp_al16(wb) || ldx % 8 || ldx < K)
    return set_error(ATMA_ERR_INVALID, "memory_gate_logits: rows must be 16-byte aligned");
  GateLogitArgs a{x, ldx, {wg, wb}, {bg, bb}, {zg, zb}, M, (int)K, (int)H};
  hipStream_t s = (hipStream_t)stream;
  return dtype == ATMA_BF16 ? launch_gate_logits<bf16>(a, s) : launch_gate_logits<f16>(a, s);
}

extern "C" int atma_polar_params_f32(const void* v_null, const void* null_base, const void* null_slope_raw,
                                     const void* len_gain_raw, const void* mag_beta_raw, float* out, int64_t H,
                                     int64_t d, int dtype, void* stream) {
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "polar_params_f32: 16-bit parameters only (dtype %d)", dtype);
  if (H < 0 || d < 1 || H * (d + 4) > 1 << 30) return set_error(ATMA_ERR_INVALID, "polar_params_f32: bad sizes");
  if (H == 0) return ATMA_OK;
  const void* p[5] = {v_null, null_base, null_slope_raw, len_gain_raw, mag_beta_raw};
  for (const void* q : p)
    if (!q || !out) return set_error(ATMA_ERR_INVALID, "polar_params_f32: null pointer");
  hipStream_t s = (hipStream_t)stream;
  return dtype == ATMA_BF16 ? launch_params<bf16>(p, out, H, d, s) : launch_params<f16>(p, out, H, d, s);
}

extern "C" int atma_paged_kv_concat(const void* k_cache, const void* v_cache, int64_t num_pages, int64_t page_size,
                                    const int32_t* pages, int64_t cached, const void* k_new, int64_t k_st,
                                    const void* v_new, int64_t v_st, int64_t n_new, void* k_out, void* v_out,
                                    int64_t row_elems, int dtype, void* stream) {
  const int es = dtype_size(dtype);
  if (!es) return set_error(ATMA_ERR_INVALID, "paged_kv_concat: unknown dtype %d", dtype);
  if (num_pages < 0 || page_size < 1 || page_size > 1 << 30 || cached < 0 || n_new < 0 || cached + n_new > 1 << 30 ||
      row_elems < 1 || row_elems > 1 << 24)
    return set_error(ATMA_ERR_INVALID, "paged_kv_concat: bad sizes");
  if (cached + n_new == 0) return ATMA_OK;
  if (!k_out || !v_out || (cached && (!k_cache || !v_cache || !pages)) || (n_new && (!k_new || !v_new)))
    return set_error(ATMA_ERR_INVALID, "paged_kv_concat: null pointer");
  if (row_elems * es % 16 || k_st * es % 16 || v_st * es % 16 || (n_new && (k_st < row_elems || v_st < row_elems)) ||
      !lp_al16(k_cache) || !lp_al16(v_cache) || !lp_al16(k_new) || !lp_al16(v_new) || !lp_al16(k_out) || !lp_al16(v_out))
    return set_error(ATMA_ERR_INVALID, "paged_kv_concat: rows must be 16-byte aligned");
  ConcatArgs a{{(const u32x4*)k_cache, (const u32x4*)v_cache}, {(const u32x4*)k_new, (const u32x4*)v_new},
               {(u32x4*)k_out, (u32x4*)v_out}, pages, cached, cached + n_new, {k_st * es / 16, v_st * es / 16},
               num_pages, (int)page_size, (int)(row_elems * es / 16)};
  const int64_t n = a.rows * a.vecs;
  kv_concat_kernel<<<dim3((unsigned)((n + 1023) / 1024), 2), dim3(256), 0, (hipStream_t)stream>>>(a);
  return check_launch("paged_kv_concat");
}
