// Training: the launches around the library GEMMs of the global block (16-bit activations, fp32 or 16-bit parameters)
// and the backwards of its elementwise parts.  Every kernel here is bound by memory: one read and one write of its
// operands.
//
// No reference counterparts as kernels: model/reference.py:22-28 (weights cast to the input's type by autograd, one GEMM
// and one bias reduction per projection), model/blocks.py:472-490 and model/reference.py:131-195 (the gates and norms),
// model/layers.py:19-31 (the MLP) run eagerly there.
#include <algorithm>

#include "common.h"

namespace atma {

__device__ __forceinline__ void load8(const void* p, int64_t i, int dt, float (&v)[8]) {
  if (dt == ATMA_F32) {
    const f32x4 a = *(const f32x4*)((const float*)p + i), b = *(const f32x4*)((const float*)p + i + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
  } else {
    const u32x4 x = *(const u32x4*)((const uint16_t*)p + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = dt == ATMA_BF16 ? elem16<bf16>(x, e) : elem16<f16>(x, e);
  }
}
__device__ __forceinline__ void store8(void* p, int64_t i, int dt, const float (&v)[8]) {
  if (dt == ATMA_F32) {
    *(f32x4*)((float*)p + i) = f32x4{v[0], v[1], v[2], v[3]};
    *(f32x4*)((float*)p + i + 4) = f32x4{v[4], v[5], v[6], v[7]};
  } else if (dt == ATMA_BF16) {
    *(u32x4*)((uint16_t*)p + i) =
        u32x4{pack2<bf16>(v[0], v[1]), pack2<bf16>(v[2], v[3]), pack2<bf16>(v[4], v[5]), pack2<bf16>(v[6], v[7])};
  } else {
    *(u32x4*)((uint16_t*)p + i) =
        u32x4{pack2<f16>(v[0], v[1]), pack2<f16>(v[2], v[3]), pack2<f16>(v[4], v[5]), pack2<f16>(v[6], v[7])};
  }
}

// ------------------------------------------------------------------ cast_blocks
// Up to 16 two-dimensional blocks converted between types and laid out anew in one launch: the parameters of several
// projections as the rows (or columns) of one GEMM operand, and that GEMM's weight gradient back as the parameters'
// own; a block of `sum` source rows of partials is summed (the bias gradients).  8 elements per thread.  (One launch
// of torch's per parameter and direction: 3 to 6 us of GPU and about 8 of host each, 26 of each in a block's step.)
constexpr int kCastBlocks = 16;
struct CastBlock {
  const void* src;
  const void* add;  // a second source like src, added, or null
  void* dst;
  int64_t sld, dld;  // elements between rows
  int rows, cols, sdt, ddt, sum;
};
struct CastArgs {
  CastBlock b[kCastBlocks];
  int first[kCastBlocks + 1];  // workgroups before
  int n;
};

__global__ void __launch_bounds__(256) cast_blocks_kernel(CastArgs a) {
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
  const CastBlock& b = a.b[i];
  const int64_t e = ((int64_t)(blockIdx.x - a.first[i]) * 256 + threadIdx.x) * 8;
  const int64_t row = e / b.cols;
  const int col = (int)(e - row * b.cols);
  if (row >= b.rows) return;
  float v[8];
  load8(b.src, row * b.sld + col, b.sdt, v);
#pragma unroll 8
  for (int p = 1; p < b.sum; ++p) {  // (partials are fp32)
    const float* w = (const float*)b.src + p * b.sld + col;
    const f32x4 x = *(const f32x4*)w, y = *(const f32x4*)(w + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += x[j], v[4 + j] += y[j];
  }
  if (b.add) {
    float w[8];
    load8(b.add, row * b.sld + col, b.sdt, w);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += w[j];
  }
  store8(b.dst, row * b.dld + col, b.ddt, v);
}

// ------------------------------------------------------------------ gather_colsum
// The gradients of one GEMM's outputs, which arrive as separate tensors, side by side as its (rows, N) operand, and each
// column's sum over kSumRows rows (fp32 partials, finished by cast_blocks): the bias gradients without another pass.
// Part p holds columns [col0[p], col0[p + 1]); with `inter` parts 0 and 1 interleave by heads of that width.  A null part
// is zeros; a null dst writes only the sums.  A workgroup takes 256 columns x kSumRows rows, a thread 8 columns.
constexpr int kGatherParts = 8, kSumRows = 128;
struct GatherArgs {
  const void* src[kGatherParts];
  int64_t ld[kGatherParts];
  int col0[kGatherParts + 1];
  int n, inter, rows, N;
  void* dst;
  float* part;
};

template <typename T>
__global__ void __launch_bounds__(256) gather_colsum_kernel(GatherArgs a) {
  __shared__ float red[8][256];
  const int cl = threadIdx.x & 31, rl = threadIdx.x >> 5;
  const int col = blockIdx.x * 256 + 8 * cl;
  const int r0 = blockIdx.y * kSumRows;
  float acc[8] = {};
  if (col < a.N) {
    int p, sc;
    if (a.inter && col < a.col0[2]) {
      const int h = col / (2 * a.inter), r = col - h * 2 * a.inter;
      p = r >= a.inter;
      sc = h * a.inter + r - p * a.inter;
    } else {
      p = a.inter ? 2 : 0;
      while (p + 1 < a.n && col >= a.col0[p + 1]) ++p;
      sc = col - a.col0[p];
    }
    const T* src = (const T*)a.src[p];
    const int64_t ld = a.ld[p];
#pragma unroll 4
    for (int i = rl; i < kSumRows; i += 8) {
      const int row = r0 + i;
      if (row >= a.rows) break;
      const u32x4 x = src ? *(const u32x4*)(src + row * ld + sc) : u32x4{0u, 0u, 0u, 0u};
      if (a.dst) *(u32x4*)((T*)a.dst + (int64_t)row * a.N + col) = x;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += elem16<T>(x, e);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[rl][8 * cl + e] = acc[e];
  __syncthreads();
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c < a.N) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 8; ++r) s += red[r][threadIdx.x];
    a.part[(int64_t)blockIdx.y * a.N + c] = s;
  }
}

// ------------------------------------------------------------------ squared_relu_gate_bwd
// h = gate relu(a)^2 with y = [a | gate]: dy = [2 gate relu(a) dh | dh relu(a)^2] (the square rounded as the forward
// rounds it), 8 columns of one row per thread.
template <typename T>
__global__ void __launch_bounds__(256) squared_relu_gate_bwd_kernel(const T* y, int64_t ldy, const T* dh, int64_t ldh, T* dy,
                                                                    int64_t rows, int W) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  const int64_t row = i / W;
  if (row >= rows) return;
  const int c = (int)(i - row * W);
  const u32x4 av = *(const u32x4*)(y + row * ldy + c), gv = *(const u32x4*)(y + row * ldy + W + c);
  const u32x4 hv = *(const u32x4*)(dh + row * ldh + c);
  float da[8], dg[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = elem16<T>(av, e), r = x > 0.f || x != x ? x : 0.f, d = elem16<T>(hv, e);
    const float sq = to_f32(from_f32<T>(r * r));
    da[e] = x > 0.f || x != x ? 2.f * r * (elem16<T>(gv, e) * d) : 0.f;
    dg[e] = sq * d;
  }
  T* o = dy + row * 2 * W + c;
  *(u32x4*)o = u32x4{pack2<T>(da[0], da[1]), pack2<T>(da[2], da[3]), pack2<T>(da[4], da[5]), pack2<T>(da[6], da[7])};
  *(u32x4*)(o + W) = u32x4{pack2<T>(dg[0], dg[1]), pack2<T>(dg[2], dg[3]), pack2<T>(dg[4], dg[5]), pack2<T>(dg[6], dg[7])};
}

// ------------------------------------------------------------------ head rows
template <int LPH>
__device__ __forceinline__ float lane_sum(float x) {  // over the LPH (8 or 16) lanes of a head
#pragma unroll
  for (int m = 1; m < LPH; m <<= 1) x += __shfl_xor(x, m, 64);
  return x;
}

// Backward of the per-head RMS norm of q and k in one launch: n = x rstd, dx = rstd (dn - n mean(dn n)).
struct HeadBwdArgs {
  const void* x[2];
  const void* dn[2];  // contiguous (rows, H, d)
  void* dx[2];        // contiguous
  int64_t ldr[2], ldh[2];
  int H[2];
  int64_t rows;
  float eps;
};

template <typename T, int LPH>
__global__ void __launch_bounds__(256) head_norm_bwd_kernel(HeadBwdArgs a) {
  constexpr int D = LPH * 8, HPW = 64 / LPH;
  const int lane = threadIdx.x & 63;
  int64_t hr = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * HPW + lane / LPH;
  const int p = hr >= a.rows * a.H[0];
  if (p) hr -= a.rows * a.H[0];
  const bool ok = hr < a.rows * a.H[p];
  if (!ok) hr = 0;
  const int64_t m = hr / a.H[p];
  const int h = (int)(hr - m * a.H[p]), e0 = 8 * (lane % LPH);
  const u32x4 xv = *(const u32x4*)((const T*)a.x[p] + m * a.ldr[p] + h * a.ldh[p] + e0);
  const u32x4 dv = *(const u32x4*)((const T*)a.dn[p] + hr * D + e0);
  float ss = 0.f, sd = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    ss = fmaf(elem16<T>(xv, e), elem16<T>(xv, e), ss);
    sd = fmaf(elem16<T>(xv, e), elem16<T>(dv, e), sd);
  }
  const float rstd = rsqrtf(lane_sum<LPH>(ss) / (float)D + a.eps);
  const float c = lane_sum<LPH>(sd) * rstd * rstd / (float)D;  // x mean(dn n) / rstd = c x
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = pack2<T>(rstd * (elem16<T>(dv, 2 * e) - c * elem16<T>(xv, 2 * e)),
                    rstd * (elem16<T>(dv, 2 * e + 1) - c * elem16<T>(xv, 2 * e + 1)));
  if (ok) *(u32x4*)((T*)a.dx[p] + hr * D + e0) = u32x4{o[0], o[1], o[2], o[3]};
}

// Backward of global_gate: xa = c sigmoid(gate), xm = round(n) sigmoid(mgate) with n = r rstd, from the gradients of
// both, side by side in dx (rows, 2 H d): dc, dgate, dmgate, dr.
struct GateBwdArgs {
  const void* c;
  int64_t c_sb, c_st, c_sh;
  int T;
  const void* gate;
  int64_t g_sr, g_sh;
  const void* r;  // contiguous (rows, H, d), T
  const void* mgate;
  int64_t mg_sr;
  const void* dx;  // contiguous (rows, 2 H d)
  void *dc, *dgate, *dr, *dmgate;  // contiguous (rows, H, d)
  int64_t rows;
  int H;
  float eps;
};

template <typename T, int LPH>
__global__ void __launch_bounds__(256) global_gate_bwd_kernel(GateBwdArgs a) {
  constexpr int D = LPH * 8, HPW = 64 / LPH;
  const int lane = threadIdx.x & 63;
  int64_t hr = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * HPW + lane / LPH;
  const bool ok = hr < a.rows * a.H;
  if (!ok) hr = 0;
  const int64_t m = hr / a.H, b = m / a.T, t = m - b * a.T;
  const int h = (int)(hr - m * a.H), e0 = 8 * (lane % LPH);
  const u32x4 cv = *(const u32x4*)((const T*)a.c + b * a.c_sb + t * a.c_st + h * a.c_sh + e0);
  const u32x4 gv = *(const u32x4*)((const T*)a.gate + m * a.g_sr + h * a.g_sh + e0);
  const u32x4 rv = *(const u32x4*)((const T*)a.r + hr * D + e0);
  const u32x4 mv = *(const u32x4*)((const T*)a.mgate + m * a.mg_sr + h * D + e0);
  const T* dx = (const T*)a.dx + m * 2 * a.H * D + h * D + e0;
  const u32x4 av = *(const u32x4*)dx, bv = *(const u32x4*)(dx + a.H * D);
  float ss = 0.f, sd = 0.f, dn[8], dc[8], dg[8], dm[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(elem16<T>(rv, e), elem16<T>(rv, e), ss);
  const float rstd = rsqrtf(lane_sum<LPH>(ss) / (float)D + a.eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float s = 1.f / (1.f + expf(-elem16<T>(gv, e))), d = elem16<T>(av, e);
    dc[e] = d * s;
    dg[e] = d * elem16<T>(cv, e) * (s * (1.f - s));
    const float sm = 1.f / (1.f + expf(-elem16<T>(mv, e))), x = elem16<T>(bv, e), r = elem16<T>(rv, e);
    dn[e] = x * sm;
    dm[e] = x * (r * rstd) * (sm * (1.f - sm));
    sd = fmaf(r, dn[e], sd);
  }
  const float k = lane_sum<LPH>(sd) * rstd * rstd / (float)D;
  if (!ok) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) dn[e] = rstd * (dn[e] - k * elem16<T>(rv, e));
  auto put = [&](void* p, const float (&v)[8]) {
    *(u32x4*)((T*)p + hr * D + e0) = u32x4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])};
  };
  put(a.dc, dc);
  put(a.dgate, dg);
  put(a.dr, dn);
  put(a.dmgate, dm);
}

static bool t_al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace atma

using namespace atma;

extern "C" int atma_cast_blocks(int n, const void* const* src, const void* const* add, void* const* dst, const int64_t* rows, const int64_t* cols,
                                const int64_t* src_ld, const int64_t* dst_ld, const int* src_dtype, const int* dst_dtype,
                                const int64_t* sum, void* stream) {
  if (n < 0 || n > kCastBlocks || (n > 0 && (!src || !dst || !rows || !cols || !src_ld || !dst_ld || !src_dtype || !dst_dtype)))
    return set_error(ATMA_ERR_INVALID, "cast_blocks: at most %d blocks", kCastBlocks);
  CastArgs a{};
  int64_t wg = 0;
  for (int i = 0; i < n; ++i) {
    if (rows[i] < 0 || cols[i] < 0 || cols[i] % 8 || rows[i] > 0x7fffffff || cols[i] > 0x7fffffff)
      return set_error(ATMA_ERR_INVALID, "cast_blocks: columns in multiples of 8");
    const int64_t s = sum ? sum[i] : 1;
    if (s < 1 || s > 0x7fffffff || (s > 1 && (rows[i] > 1 || src_dtype[i] != ATMA_F32)))
      return set_error(ATMA_ERR_INVALID, "cast_blocks: sums of one row of fp32 partials");
    for (int dt : {src_dtype[i], dst_dtype[i]})
      if (dt != ATMA_F32 && dt != ATMA_BF16 && dt != ATMA_F16)
        return set_error(ATMA_ERR_UNSUPPORTED, "cast_blocks: unknown dtype %d", dt);
    if (rows[i] == 0 || cols[i] == 0) continue;
    if (!src[i] || !dst[i] || !t_al16(src[i]) || (add && !t_al16(add[i])) || !t_al16(dst[i]) || src_ld[i] % 8 || dst_ld[i] % 8)
      return set_error(ATMA_ERR_INVALID, "cast_blocks: 16-byte aligned rows");
    a.b[a.n] = CastBlock{src[i], add ? add[i] : nullptr, dst[i], src_ld[i], dst_ld[i], (int)rows[i], (int)cols[i], src_dtype[i], dst_dtype[i], (int)s};
    a.first[a.n++] = (int)wg;
    wg += (rows[i] * cols[i] + 2047) / 2048;
    if (wg > 0x7fffffff) return set_error(ATMA_ERR_INVALID, "cast_blocks: sizes too large");
  }
  if (a.n == 0) return ATMA_OK;
  a.first[a.n] = (int)wg;
  cast_blocks_kernel<<<dim3((unsigned)wg), dim3(256), 0, (hipStream_t)stream>>>(a);
  return check_launch("cast_blocks");
}

extern "C" size_t atma_gather_colsum_partials(int64_t rows) {
  return rows > 0 ? (size_t)((rows + kSumRows - 1) / kSumRows) : 0;
}

extern "C" int atma_gather_colsum(int n, const void* const* src, const int64_t* ld, const int64_t* width, int64_t inter,
                                  void* dst, float* part, int64_t rows, int dtype, void* stream) {
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "gather_colsum: 16-bit only (dtype %d)", dtype);
  if (n < 1 || n > kGatherParts || !src || !ld || !width || rows < 0 || rows > 0x7fffffff || inter < 0 || inter % 8 ||
      (inter && (n < 2 || width[0] != width[1] || width[0] % inter)))
    return set_error(ATMA_ERR_INVALID, "gather_colsum: bad parts");
  GatherArgs a{};
  int64_t N = 0;
  for (int i = 0; i < n; ++i) {
    if (width[i] < 8 || width[i] % 8 || ld[i] % 8 || !t_al16(src[i]) || N + width[i] > 0x7fffffff - 256)
      return set_error(ATMA_ERR_INVALID, "gather_colsum: widths in multiples of 8, 16-byte aligned rows");
    a.src[i] = src[i];
    a.ld[i] = ld[i];
    a.col0[i] = (int)N;
    N += width[i];
  }
  a.col0[n] = (int)N;
  if (rows == 0) return ATMA_OK;
  if (!part || (uintptr_t)part % 4 || !t_al16(dst)) return set_error(ATMA_ERR_INVALID, "gather_colsum: null or misaligned pointer");
  const int64_t chunks = (rows + kSumRows - 1) / kSumRows;
  if (chunks > 65535) return set_error(ATMA_ERR_UNSUPPORTED, "gather_colsum: too many rows");
  a.n = n; a.inter = (int)inter; a.rows = (int)rows; a.N = (int)N; a.dst = dst; a.part = part;
  const dim3 grid((unsigned)((N + 255) / 256), (unsigned)chunks);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_BF16) gather_colsum_kernel<bf16><<<grid, dim3(256), 0, s>>>(a);
  else gather_colsum_kernel<f16><<<grid, dim3(256), 0, s>>>(a);
  return check_launch("gather_colsum");
}

extern "C" int atma_squared_relu_gate_bwd(const void* y, int64_t ldy, const void* dh, int64_t ldh, void* dy, int64_t rows,
                                          int64_t width, int dtype, void* stream) {
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "squared_relu_gate_bwd: 16-bit only (dtype %d)", dtype);
  if (rows < 0 || width < 8 || width % 8 || width > 0x3fffffff || ldy % 8 || ldh % 8 || ldy < 2 * width || ldh < 0 ||
      rows > ((int64_t)1 << 40) / width)
    return set_error(ATMA_ERR_INVALID, "squared_relu_gate_bwd: bad sizes");
  if (rows == 0) return ATMA_OK;
  if (!y || !dh || !dy || !t_al16(y) || !t_al16(dh) || !t_al16(dy))
    return set_error(ATMA_ERR_INVALID, "squared_relu_gate_bwd: null or misaligned pointer");
  const int64_t wg = (rows * width + 2047) / 2048;
  if (wg > 0x7fffffff) return set_error(ATMA_ERR_INVALID, "squared_relu_gate_bwd: sizes too large");
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_BF16)
    squared_relu_gate_bwd_kernel<bf16><<<dim3((unsigned)wg), dim3(256), 0, s>>>((const bf16*)y, ldy, (const bf16*)dh, ldh,
                                                                                (bf16*)dy, rows, (int)width);
  else
    squared_relu_gate_bwd_kernel<f16><<<dim3((unsigned)wg), dim3(256), 0, s>>>((const f16*)y, ldy, (const f16*)dh, ldh,
                                                                               (f16*)dy, rows, (int)width);
  return check_launch("squared_relu_gate_bwd");
}

extern "C" int atma_head_norm_bwd(const void* const* x, const int64_t* ldr, const int64_t* ldh, const int64_t* heads,
                                  const void* const* dn, void* const* dx, int64_t rows, int64_t d, float eps, int dtype,
                                  void* stream) {
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "head_norm_bwd: 16-bit only (dtype %d)", dtype);
  if (!x || !ldr || !ldh || !heads || !dn || !dx || rows < 0 || (d != 64 && d != 128) || rows > (int64_t)1 << 40)
    return set_error(ATMA_ERR_INVALID, "head_norm_bwd: bad sizes (d 64 or 128)");
  HeadBwdArgs a{};
  int64_t hr = 0;
  for (int p = 0; p < 2; ++p) {
    if (heads[p] < 1 || heads[p] > 4096 || ldr[p] % 8 || ldh[p] % 8)
      return set_error(ATMA_ERR_INVALID, "head_norm_bwd: bad heads");
    if (rows > 0 && (!x[p] || !dn[p] || !dx[p] || !t_al16(x[p]) || !t_al16(dn[p]) || !t_al16(dx[p])))
      return set_error(ATMA_ERR_INVALID, "head_norm_bwd: null or misaligned pointer");
    a.x[p] = x[p]; a.dn[p] = dn[p]; a.dx[p] = dx[p]; a.ldr[p] = ldr[p]; a.ldh[p] = ldh[p]; a.H[p] = (int)heads[p];
    hr += rows * heads[p];
  }
  if (rows == 0) return ATMA_OK;
  a.rows = rows; a.eps = eps;
  const int64_t per = 4 * 64 / (d / 8), wg = (hr + per - 1) / per;
  if (wg > 0x7fffffff) return set_error(ATMA_ERR_INVALID, "head_norm_bwd: sizes too large");
  const dim3 grid((unsigned)wg);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_BF16) {
    if (d == 128) head_norm_bwd_kernel<bf16, 16><<<grid, dim3(256), 0, s>>>(a);
    else head_norm_bwd_kernel<bf16, 8><<<grid, dim3(256), 0, s>>>(a);
  } else {
    if (d == 128) head_norm_bwd_kernel<f16, 16><<<grid, dim3(256), 0, s>>>(a);
    else head_norm_bwd_kernel<f16, 8><<<grid, dim3(256), 0, s>>>(a);
  }
  return check_launch("head_norm_bwd");
}

extern "C" int atma_global_gate_bwd(const void* c, int64_t c_sb, int64_t c_st, int64_t c_sh, int64_t T, const void* gate,
                                    int64_t g_sr, int64_t g_sh, const void* r, const void* mgate, int64_t mg_sr,
                                    const void* dx, void* dc, void* dgate, void* dr, void* dmgate, int64_t rows, int64_t H,
                                    int64_t d, float eps, int dtype, void* stream) {
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "global_gate_bwd: 16-bit only (dtype %d)", dtype);
  if (rows < 0 || H < 1 || H > 4096 || (d != 64 && d != 128) || T < 1 || T > 0x7fffffff || rows % T || rows > (int64_t)1 << 40)
    return set_error(ATMA_ERR_INVALID, "global_gate_bwd: bad sizes (d 64 or 128, rows a multiple of T)");
  if (rows == 0) return ATMA_OK;
  if (!c || !gate || !r || !mgate || !dx || !dc || !dgate || !dr || !dmgate || !t_al16(c) || !t_al16(gate) || !t_al16(r) ||
      !t_al16(mgate) || !t_al16(dx) || !t_al16(dc) || !t_al16(dgate) || !t_al16(dr) || !t_al16(dmgate) || c_sb % 8 ||
      c_st % 8 || c_sh % 8 || g_sr % 8 || g_sh % 8 || mg_sr % 8)
    return set_error(ATMA_ERR_INVALID, "global_gate_bwd: null or misaligned pointer");
  GateBwdArgs a{c, c_sb, c_st, c_sh, (int)T, gate, g_sr, g_sh, r, mgate, mg_sr, dx, dc, dgate, dr, dmgate, rows, (int)H, eps};
  const int64_t per = 4 * 64 / (d / 8), wg = (rows * H + per - 1) / per;
  if (wg > 0x7fffffff) return set_error(ATMA_ERR_INVALID, "global_gate_bwd: sizes too large");
  const dim3 grid((unsigned)wg);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_BF16) {
    if (d == 128) global_gate_bwd_kernel<bf16, 16><<<grid, dim3(256), 0, s>>>(a);
    else global_gate_bwd_kernel<bf16, 8><<<grid, dim3(256), 0, s>>>(a);
  } else {
    if (d == 128) global_gate_bwd_kernel<f16, 16><<<grid, dim3(256), 0, s>>>(a);
    else global_gate_bwd_kernel<f16, 8><<<grid, dim3(256), 0, s>>>(a);
  }
  return check_launch("global_gate_bwd");
}
