// The global layer's Canon step on whole rows: per-head RMSNorm of q and k, the residual causal depthwise conv
// of q, k and v (model/reference.py:136-155; the engine's tails inference/models/atma.py:102-162), the convs'
// state rows and the K/V rows of the paged cache, in one launch; and the conv's training backward.
//
//  * canon_fwd: with xn = norm ? round(rms_norm(x)) : x per head-row, out[t] = round(xn[t] + sum_j w[j] xn[t - (K-1) + j]),
//    the sum in fp32 (eager torch rounds the conv before the add, so this is the better-rounded form).  Rows before a
//    sequence's start are zero, or its stored tail when the call continues a sequence.
//  * canon_bwd: dx[t] = round(dy[t] + sum_j w[j] dy[t + (K-1) - j]), dw[c][j] = sum_t dy[t][c] x[t - (K-1) + j][c]
//    in fp32: each strip's partial sums, then one reduction in a fixed order (deterministic).
//
// Both are HBM streams.  A head-row of d values is d / 8 lanes of 8 (16-byte loads for 16-bit types), so the norm is a
// DPP row sum; a lane walks a strip of tokens with the K - 1 previous rows in registers and loads 8 rows ahead of their
// arithmetic.  Strips are 32 tokens where that still gives two waves to every SIMD, else 16 or 8: a short prompt is
// bound by its loads' latency, and the K - 1 rows a strip reads twice cost less than idle CUs.
//
// Measured (8 / 2 heads, d = 128, K = 4, bf16): 65,536 rows 88 us (403 MB, 4.6 TB/s) where the eager chain (two norms, three
// library depthwise convs with their padding and transposes, three adds) took about 3.0 ms; 2,999 rows 14 us against
// about 75 us.  In training (5,700 rows) the library convs and their backward took about 2.2 ms of a block's 4.1 ms.
#include "common.h"

namespace atma {

constexpr int kCanonRows = 8;  // rows a lane loads before it works on them

struct CanonStream {
  const void* x;  // element (row, head, e) at row ldr + head ldh + e
  int64_t ldr, ldh;
  const void* w;  // (H d, K) contiguous
  void* out;      // (rows, H, d) contiguous
  void* tails;    // (num_slots, H d, K - 1), row stride t_ss; or null
  int64_t t_ss;
  void* cache;  // (total_slots, H, d) contiguous; or null
  int H, norm;
};

struct CanonArgs {
  CanonStream s[3];
  int heads;  // of all streams
  int64_t rows, T;  // T > 0: rows / T sequences of T rows; 0: the token maps
  const int32_t *seq_start, *seq_end, *seq_slot;
  const int64_t* slots;  // (rows / T) table rows, or null
  int64_t num_slots;
  int continuing;
  const int32_t* slot_map;  // (rows) cache rows, or null
  int64_t total_slots;
  float eps;
  int strip, per_seq;  // tokens of a strip; strips of a sequence (T > 0)
  int64_t strips;
};

template <int LPH>
__device__ __forceinline__ float canon_head_sum(float x) {
  x += dpp_f32<0xB1>(x);
  x += dpp_f32<0x4E>(x);
  x += dpp_f32<0x141>(x);
  if constexpr (LPH == 16) x += dpp_f32<0x140>(x);
  return x;
}

// 8 consecutive elements.
template <typename T>
struct Row8 {
  u32x4 u;
  __device__ __forceinline__ void load(const T* p) { u = *(const u32x4*)p; }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = elem16<T>(u, e);
  }
  __device__ __forceinline__ void put(const float* v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = pack2<T>(v[2 * e], v[2 * e + 1]);
  }
  __device__ __forceinline__ void store(T* p) const { *(u32x4*)p = u; }
};
template <>
struct Row8<float> {
  f32x4 u[2];
  __device__ __forceinline__ void load(const float* p) { u[0] = *(const f32x4*)p, u[1] = *(const f32x4*)(p + 4); }
  __device__ __forceinline__ void get(float* v) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = u[e >> 2][e & 3];
  }
  __device__ __forceinline__ void put(const float* v) {
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e >> 2][e & 3] = v[e];
  }
  __device__ __forceinline__ void store(float* p) const { *(f32x4*)p = u[0], *(f32x4*)(p + 4) = u[1]; }
};

// The 8 K taps of a lane's 8 channels: 8 K consecutive elements, read as K groups of 8.
template <typename TW, int K>
__device__ __forceinline__ void canon_taps(const TW* w, float (*wt)[8]) {
  float f[8 * K];
  Row8<TW> r[K];
#pragma unroll
  for (int i = 0; i < K; ++i) r[i].load(w + 8 * i);
#pragma unroll
  for (int i = 0; i < K; ++i) r[i].get(f + 8 * i);
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int j = 0; j < K; ++j) wt[j][e] = f[e * K + j];
}

template <typename T, typename TW, int LPH, int K>
__global__ void __launch_bounds__(256) canon_fwd_kernel(CanonArgs a) {
  constexpr int D = LPH * 8, HPW = 64 / LPH;
  const int lane = threadIdx.x & 63;
  const int64_t strip = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int hg = blockIdx.y * HPW + lane / LPH;
  if (strip >= a.strips || hg >= a.heads) return;  // whole head-rows drop out: the DPP sums stay whole
  const int h0 = a.s[0].H, h1 = h0 + a.s[1].H;
  const int si = hg < h0 ? 0 : hg < h1 ? 1 : 2;
  auto pick = [&](auto f) { return si == 0 ? f(a.s[0]) : si == 1 ? f(a.s[1]) : f(a.s[2]); };
  const int h = hg - (si == 0 ? 0 : si == 1 ? h0 : h1);
  const int H = pick([](const CanonStream& s) { return s.H; });
  const bool norm = pick([](const CanonStream& s) { return s.norm; }) != 0;
  const int64_t ldr = pick([](const CanonStream& s) { return s.ldr; });
  const int e0 = 8 * (lane % LPH);
  const int64_t c0 = (int64_t)h * D + e0;  // the lane's first channel in its stream
  const T* x = (const T*)pick([](const CanonStream& s) { return s.x; }) +
               h * pick([](const CanonStream& s) { return s.ldh; }) + e0;
  T* out = (T*)pick([](const CanonStream& s) { return s.out; }) + c0;
  T* tails = (T*)pick([](const CanonStream& s) { return s.tails; });
  T* cache = (T*)pick([](const CanonStream& s) { return s.cache; });
  const int64_t t_ss = pick([](const CanonStream& s) { return s.t_ss; });
  const int64_t ldo = (int64_t)H * D;

  const bool dense = a.T > 0;
  const int64_t seq = dense ? strip / a.per_seq : 0;
  const int64_t seq_beg = seq * a.T, seq_end = dense ? seq_beg + a.T : a.rows;
  const int64_t t_beg = dense ? seq_beg + (strip - seq * a.per_seq) * a.strip : strip * a.strip;
  const int64_t t_end = min(t_beg + a.strip, seq_end);

  float wt[K][8];
  canon_taps<TW, K>((const TW*)pick([](const CanonStream& s) { return s.w; }) + c0 * K, wt);
  auto normed = [&](float* v) {  // round(rms_norm(v)) over the head-row
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
    const float rstd = rsqrtf(canon_head_sum<LPH>(ss) / (float)D + a.eps);
    if (norm) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = to_f32(from_f32<T>(v[e] * rstd));
    }
  };
  auto row = [&](int64_t t, float* v) {
    Row8<T> r;
    r.load(x + t * ldr);
    r.get(v);
    normed(v);
  };

  float win[K][8];
  const bool first = dense && t_beg == seq_beg;
  int64_t slot = -1;
  if (first && tails && a.slots) {
    slot = a.slots[seq];
    if (a.continuing && slot < 0) slot += a.num_slots;  // a row counted from the end, as the memory's state beside it
  }
  if (slot >= a.num_slots) slot = -1;
  if (first) {
#pragma unroll
    for (int j = 0; j < K - 1; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        win[j][e] = a.continuing && slot >= 0 ? to_f32(tails[slot * t_ss + (c0 + e) * (K - 1) + j]) : 0.f;
    if (slot >= 0) {
      // the sequence's last K - 1 inputs become its stored tail: written here, by the lane that has just read the
      // old one, and not by the last strip, which may run before this one
#pragma unroll
      for (int j = 0; j < K - 1; ++j) {
        const int64_t t = seq_end - (K - 1) + j;
        float v[8];
        if (t >= seq_beg) {
          row(t, v);
        } else {  // a chunk shorter than the tail keeps what remains of it
#pragma unroll
          for (int i = 0; i < K - 1; ++i)
            if (i == a.T + j) {
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] = win[i][e];
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) tails[slot * t_ss + (c0 + e) * (K - 1) + j] = from_f32<T>(v[e]);
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < K - 1; ++j) {
      const int64_t t = t_beg - (K - 1) + j;
      if (t >= seq_beg) {
        row(t, win[j]);
      } else {  // a strip shorter than the taps' reach is never second; packed rows before the first are masked below
#pragma unroll
        for (int e = 0; e < 8; ++e) win[j][e] = 0.f;
      }
    }
  }

  for (int64_t tb = t_beg; tb < t_end; tb += kCanonRows) {
    Row8<T> raw[kCanonRows];
#pragma unroll
    for (int u = 0; u < kCanonRows; ++u) raw[u].load(x + min(tb + u, t_end - 1) * ldr);
#pragma unroll
    for (int u = 0; u < kCanonRows; ++u) {
      const int64_t t = tb + u;
      if (t < t_end) {
        raw[u].get(win[K - 1]);
        normed(win[K - 1]);
        const int64_t start = dense ? seq_beg : (int64_t)a.seq_start[t];
        float acc[8], o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll
        for (int j = 0; j < K; ++j) {
          const bool live = dense || t - (K - 1 - j) >= start;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] = fmaf(live ? win[j][e] : 0.f, wt[j][e], acc[e]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = win[K - 1][e] + acc[e];
        Row8<T> r;
        r.put(o);
        r.store(out + t * ldo);
        if (cache) {
          const int64_t cs = a.slot_map[t];
          if (cs >= 0 && cs < a.total_slots) r.store(cache + cs * ldo + c0);
        }
        if (!dense && tails && t == (int64_t)a.seq_end[t] - 1) {
          const int64_t sl = a.seq_slot[t];
          if (sl >= 0 && sl < a.num_slots) {
#pragma unroll
            for (int j = 0; j < K - 1; ++j) {
              const bool live = t - (K - 2 - j) >= start;
#pragma unroll
              for (int e = 0; e < 8; ++e)
                tails[sl * t_ss + (c0 + e) * (K - 1) + j] = from_f32<T>(live ? win[j + 1][e] : 0.f);
            }
          }
        }
#pragma unroll
        for (int j = 0; j < K - 1; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) win[j][e] = win[j + 1][e];
      }
    }
  }
}

// ------------------------------------------------------------------ backward
struct CanonBwdStream {
  const void *dy, *x;  // (rows, C) contiguous
  const void* w;       // (C, K)
  void* dx;            // (rows, C)
  float* part;         // (strips, C, K)
  void* dw;            // (C, K)
  int C;
};

struct CanonBwdArgs {
  CanonBwdStream s[3];
  int groups;  // 8-channel groups of all streams
  int64_t rows, T;
  int strip, per_seq;
  int64_t strips;
};

template <typename T, typename TW, int K>
__global__ void __launch_bounds__(256) canon_bwd_kernel(CanonBwdArgs a) {
  const int g = blockIdx.y * 64 + (threadIdx.x & 63);
  const int64_t strip = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= a.groups || strip >= a.strips) return;
  const int g0 = a.s[0].C / 8, g1 = g0 + a.s[1].C / 8;
  const int si = g < g0 ? 0 : g < g1 ? 1 : 2;
  auto pick = [&](auto f) { return si == 0 ? f(a.s[0]) : si == 1 ? f(a.s[1]) : f(a.s[2]); };
  const int64_t C = pick([](const CanonBwdStream& s) { return s.C; });
  const int64_t c0 = 8 * (int64_t)(g - (si == 0 ? 0 : si == 1 ? g0 : g1));
  const T* dy = (const T*)pick([](const CanonBwdStream& s) { return s.dy; }) + c0;
  const T* x = (const T*)pick([](const CanonBwdStream& s) { return s.x; }) + c0;
  T* dx = (T*)pick([](const CanonBwdStream& s) { return s.dx; }) + c0;
  float* part = pick([](const CanonBwdStream& s) { return s.part; }) + (strip * C + c0) * K;
  float wt[K][8];
  canon_taps<TW, K>((const TW*)pick([](const CanonBwdStream& s) { return s.w; }) + c0 * K, wt);

  const int64_t seq = strip / a.per_seq;
  const int64_t seq_beg = seq * a.T, seq_end = seq_beg + a.T;
  const int64_t t_beg = seq_beg + (strip - seq * a.per_seq) * a.strip, t_end = min(t_beg + a.strip, seq_end);
  auto row = [&](const T* p, int64_t t, float* v) {  // row t of the sequence, zero outside it
    if (t >= seq_beg && t < seq_end) {
      Row8<T> r;
      r.load(p + t * C);
      r.get(v);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
    }
  };
  float dw[K][8], xw[K][8], gw[K][8];  // x rows t - (K-1) .. t, dy rows t .. t + K - 1
#pragma unroll
  for (int j = 0; j < K; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) dw[j][e] = 0.f;
#pragma unroll
  for (int j = 0; j < K - 1; ++j) {
    row(x, t_beg - (K - 1) + j, xw[j]);
    row(dy, t_beg + j, gw[j]);
  }
  for (int64_t tb = t_beg; tb < t_end; tb += kCanonRows) {
    Row8<T> rx[kCanonRows], rg[kCanonRows];
#pragma unroll
    for (int u = 0; u < kCanonRows; ++u) {
      rx[u].load(x + min(tb + u, seq_end - 1) * C);
      rg[u].load(dy + min(tb + u + K - 1, seq_end - 1) * C);
    }
#pragma unroll
    for (int u = 0; u < kCanonRows; ++u) {
      const int64_t t = tb + u;
      if (t < t_end) {
        rx[u].get(xw[K - 1]);
        rg[u].get(gw[K - 1]);
        if (t + K - 1 >= seq_end) {
#pragma unroll
          for (int e = 0; e < 8; ++e) gw[K - 1][e] = 0.f;
        }
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = 0.f;
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            o[e] = fmaf(wt[j][e], gw[K - 1 - j][e], o[e]);
            dw[j][e] = fmaf(gw[0][e], xw[j][e], dw[j][e]);
          }
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] += gw[0][e];
        Row8<T> r;
        r.put(o);
        r.store(dx + t * C);
#pragma unroll
        for (int j = 0; j < K - 1; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            xw[j][e] = xw[j + 1][e];
            gw[j][e] = gw[j + 1][e];
          }
      }
    }
  }
  float f[8 * K];
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int j = 0; j < K; ++j) f[e * K + j] = dw[j][e];
#pragma unroll
  for (int i = 0; i < 2 * K; ++i) *(f32x4*)(part + 4 * i) = (f32x4){f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]};
}

// dw = the strips' partial sums, 16 slices of the strips at a time and then the slices, both in a fixed order.
template <typename TW>
__global__ void __launch_bounds__(256) canon_dw_kernel(CanonBwdArgs a, int K) {
  __shared__ f32x4 sum[16][16];
  const int64_t col = (int64_t)blockIdx.x * 16 + (threadIdx.x & 15);  // 4 taps of a stream
  const int64_t n0 = (int64_t)a.s[0].C * K / 4, n1 = n0 + (int64_t)a.s[1].C * K / 4;
  const int64_t n2 = n1 + (int64_t)a.s[2].C * K / 4;
  const int si = col < n0 ? 0 : col < n1 ? 1 : 2;
  auto pick = [&](auto f) { return si == 0 ? f(a.s[0]) : si == 1 ? f(a.s[1]) : f(a.s[2]); };
  const int64_t i = 4 * (col - (si == 0 ? 0 : si == 1 ? n0 : n1));
  const int64_t CK = pick([](const CanonBwdStream& s) { return (int64_t)s.C; }) * K;
  const float* part = pick([](const CanonBwdStream& s) { return (const float*)s.part; });
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (col < n2)
    for (int64_t s = threadIdx.x >> 4; s < a.strips; s += 16) acc += *(const f32x4*)(part + s * CK + i);
  sum[threadIdx.x >> 4][threadIdx.x & 15] = acc;
  __syncthreads();
  if (threadIdx.x < 16 && col < n2) {
#pragma unroll
    for (int s = 1; s < 16; ++s) acc += sum[s][threadIdx.x];
    TW* dw = (TW*)pick([](const CanonBwdStream& s) { return s.dw; }) + i;
#pragma unroll
    for (int e = 0; e < 4; ++e) dw[e] = from_f32<TW>(acc[e]);
  }
}

// Tokens of a strip: 32 where that leaves two waves for each SIMD of the device, else 16, else 8.
static int canon_strip(int64_t seqs, int64_t T, int64_t col_waves) {
  const int64_t want = 8 * (int64_t)device_cu_count();
  for (int s = 32; s > 8; s /= 2)
    if (seqs * ((T + s - 1) / s) * col_waves >= want) return s;
  return 8;
}

static bool canon_al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

template <typename T, typename TW>
static int launch_canon(const CanonArgs& a, int64_t K, int64_t d, hipStream_t s) {
  const dim3 grid((unsigned)((a.strips + 3) / 4), (unsigned)((a.heads + 512 / d - 1) / (512 / d)));
#define ATMA_CANON(LPH, KK) canon_fwd_kernel<T, TW, LPH, KK><<<grid, dim3(256), 0, s>>>(a)
  if (d == 128) {
    if (K == 2) ATMA_CANON(16, 2);
    else if (K == 3) ATMA_CANON(16, 3);
    else ATMA_CANON(16, 4);
  } else {
    if (K == 2) ATMA_CANON(8, 2);
    else if (K == 3) ATMA_CANON(8, 3);
    else ATMA_CANON(8, 4);
  }
#undef ATMA_CANON
  return check_launch("canon_qkv");
}

template <typename T, typename TW>
static int launch_canon_bwd(const CanonBwdArgs& a, int64_t K, hipStream_t s) {
  const dim3 grid((unsigned)((a.strips + 3) / 4), (unsigned)((a.groups + 63) / 64));
  if (K == 2) canon_bwd_kernel<T, TW, 2><<<grid, dim3(256), 0, s>>>(a);
  else if (K == 3) canon_bwd_kernel<T, TW, 3><<<grid, dim3(256), 0, s>>>(a);
  else canon_bwd_kernel<T, TW, 4><<<grid, dim3(256), 0, s>>>(a);
  const int64_t cols = (int64_t)a.groups * 2 * K;
  canon_dw_kernel<TW><<<dim3((unsigned)((cols + 15) / 16)), dim3(256), 0, s>>>(a, (int)K);
  return check_launch("canon_bwd");
}

}  // namespace atma

using namespace atma;

extern "C" int atma_canon_qkv(const void* const* x, const int64_t* ldr, const int64_t* ldh, const int64_t* heads,
                              const int* norm, const void* const* w, void* const* out, void* const* tails,
                              const int64_t* tails_ss, void* const* cache, int64_t n, int64_t rows, int64_t T,
                              const int32_t* seq_starts, const int32_t* seq_ends, const int32_t* seq_slots,
                              const int64_t* slots, int64_t num_slots, int continuing, const int32_t* slot_mapping,
                              int64_t total_slots, int64_t K, int64_t d, float eps, int w_dtype, int dtype,
                              void* stream) {
  const int es = dtype_size(dtype);
  if (!es || (w_dtype != dtype && w_dtype != ATMA_F32))
    return set_error(ATMA_ERR_INVALID, "canon_qkv: weights in the rows' dtype or fp32");
  if (K < 2 || K > 4 || (d != 64 && d != 128))
    return set_error(ATMA_ERR_UNSUPPORTED, "canon_qkv: kernel size %lld, head width %lld (2..4; 64 or 128)", (long long)K,
                     (long long)d);
  if (n < 1 || n > 3 || rows < 0 || rows > 0x7fffffff || T < 0 || (T && rows % T) || num_slots < 0 || total_slots < 0)
    return set_error(ATMA_ERR_INVALID, "canon_qkv: bad sizes");
  if (rows == 0) return ATMA_OK;
  if (!x || !ldr || !ldh || !heads || !norm || !w || !out)
    return set_error(ATMA_ERR_INVALID, "canon_qkv: null pointer");
  CanonArgs a{};
  bool any_tails = false;
  for (int i = 0; i < n; ++i) {
    CanonStream& s = a.s[i];
    s = CanonStream{x[i], ldr[i], ldh[i], w[i], out[i], tails ? tails[i] : nullptr, tails ? tails_ss[i] : 0,
                    cache ? cache[i] : nullptr, (int)heads[i], norm[i]};
    if (heads[i] < 1 || heads[i] > 1 << 16 || !s.x || !s.w || !s.out)
      return set_error(ATMA_ERR_INVALID, "canon_qkv: bad stream");
    if (!canon_al16(s.x) || !canon_al16(s.w) || !canon_al16(s.out) || !canon_al16(s.cache) || ldr[i] * es % 16 ||
        ldh[i] * es % 16 || ldh[i] < d || ldr[i] < ldh[i] * (heads[i] - 1) + d)
      return set_error(ATMA_ERR_INVALID, "canon_qkv: head-rows must be 16-byte aligned and not overlap");
    if (s.cache && !slot_mapping) return set_error(ATMA_ERR_INVALID, "canon_qkv: cache without slot_mapping");
    if (s.tails && s.t_ss < heads[i] * d * (K - 1)) return set_error(ATMA_ERR_INVALID, "canon_qkv: tails overlap");
    any_tails |= s.tails != nullptr;
    a.heads += (int)heads[i];
  }
  if (!T && (!seq_starts || (any_tails && (!seq_ends || !seq_slots)) || continuing))
    return set_error(ATMA_ERR_INVALID, "canon_qkv: packed rows need their maps and start fresh");
  if (T && any_tails && !slots) return set_error(ATMA_ERR_INVALID, "canon_qkv: tails without slots");
  if (continuing && !any_tails) return set_error(ATMA_ERR_INVALID, "canon_qkv: nothing to continue from");
  a.rows = rows, a.T = T;
  a.seq_start = seq_starts, a.seq_end = seq_ends, a.seq_slot = seq_slots, a.slots = slots, a.num_slots = num_slots;
  a.continuing = continuing, a.slot_map = slot_mapping, a.total_slots = total_slots, a.eps = eps;
  const int64_t len = T ? T : rows;
  a.strip = canon_strip(rows / len, len, (a.heads + 512 / d - 1) / (512 / d));
  a.per_seq = (int)((len + a.strip - 1) / a.strip);
  a.strips = rows / len * a.per_seq;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_F32) return launch_canon<float, float>(a, K, d, s);
  if (dtype == ATMA_BF16)
    return w_dtype == ATMA_F32 ? launch_canon<bf16, float>(a, K, d, s) : launch_canon<bf16, bf16>(a, K, d, s);
  return w_dtype == ATMA_F32 ? launch_canon<f16, float>(a, K, d, s) : launch_canon<f16, f16>(a, K, d, s);
}

extern "C" size_t atma_canon_bwd_workspace_bytes(int64_t rows, int64_t T, int64_t channels, int64_t K) {
  if (rows <= 0 || T <= 0 || channels <= 0 || K <= 0) return 0;
  const int64_t strip = canon_strip(rows / T, T, (channels / 8 + 63) / 64);
  return (size_t)(rows / T * ((T + strip - 1) / strip) * channels * K) * 4;
}

extern "C" int atma_canon_bwd(const void* const* dy, const void* const* x, const void* const* w, void* const* dx,
                              void* const* dw, const int64_t* channels, int64_t n, int64_t rows, int64_t T, int64_t K,
                              int w_dtype, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  if (!dtype_size(dtype) || (w_dtype != dtype && w_dtype != ATMA_F32))
    return set_error(ATMA_ERR_INVALID, "canon_bwd: weights in the rows' dtype or fp32");
  if (K < 2 || K > 4) return set_error(ATMA_ERR_UNSUPPORTED, "canon_bwd: kernel size %lld (2..4)", (long long)K);
  if (n < 1 || n > 3 || rows < 1 || rows > 0x7fffffff || T < 1 || rows % T)
    return set_error(ATMA_ERR_INVALID, "canon_bwd: bad sizes");
  if (!dy || !x || !w || !dx || !dw || !channels || !workspace)
    return set_error(ATMA_ERR_INVALID, "canon_bwd: null pointer");
  int64_t total = 0;
  for (int i = 0; i < n; ++i) {
    if (channels[i] < 8 || channels[i] % 8 || channels[i] > 1 << 24)
      return set_error(ATMA_ERR_INVALID, "canon_bwd: channels must be a multiple of 8");
    if (!canon_al16(dy[i]) || !canon_al16(x[i]) || !canon_al16(w[i]) || !canon_al16(dx[i]) || !dy[i] || !x[i] || !w[i] ||
        !dx[i] || !dw[i])
      return set_error(ATMA_ERR_INVALID, "canon_bwd: rows must be 16-byte aligned");
    total += channels[i];
  }
  if (workspace_bytes < atma_canon_bwd_workspace_bytes(rows, T, total, K) || !canon_al16(workspace))
    return set_error(ATMA_ERR_WORKSPACE, "canon_bwd: workspace too small");
  CanonBwdArgs a{};
  a.rows = rows, a.T = T;
  a.strip = canon_strip(rows / T, T, (total / 8 + 63) / 64);
  a.per_seq = (int)((T + a.strip - 1) / a.strip);
  a.strips = rows / T * a.per_seq;
  float* part = (float*)workspace;
  for (int i = 0; i < n; ++i) {
    a.s[i] = CanonBwdStream{dy[i], x[i], w[i], dx[i], part, dw[i], (int)channels[i]};
    part += a.strips * channels[i] * K;
    a.groups += (int)(channels[i] / 8);
  }
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_F32) return launch_canon_bwd<float, float>(a, K, s);
  if (dtype == ATMA_BF16)
    return w_dtype == ATMA_F32 ? launch_canon_bwd<bf16, float>(a, K, s) : launch_canon_bwd<bf16, bf16>(a, K, s);
  return w_dtype == ATMA_F32 ? launch_canon_bwd<f16, float>(a, K, s) : launch_canon_bwd<f16, f16>(a, K, s);
}
