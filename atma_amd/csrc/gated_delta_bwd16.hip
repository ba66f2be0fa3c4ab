// Chunked backward of the gated-delta recurrence for 16-bit training: the sequential part.
//
// Reference: the memory branch trains through FLA's chunk_gated_delta_rule autograd
// (model/blocks.py:44-84); the recurrence is scripts/titans_proto.py:53-76 in the [K, V]
// layout.  Inside a 64-token chunk with inclusive log decays lg, Ga = exp(lg),
// w = exp(lg_C - lg), T = (I + diag(beta) A)^-1 (A[p,s] = exp(lg_p - lg_s) k_p.k_s, s < p)
// and Rq[p,s] = exp(lg_p - lg_s) q_p.k_s (s <= p), the forward is
//   U = T diag(beta) (V - diag(Ga) K S),   S' = Ga_C S + K^T diag(w) U,
// and the backward carries dS = dL/dS' from the last chunk to the first:
//   dU = Rq^T dO + diag(w) K dS,   dY = T^T dU,
//   dS <- Ga_C dS + Q^T diag(Ga) dO - K^T diag(Ga beta) dY.
// This kernel runs both chains (the forward one to recover each chunk's entry state
// and the backward one, which do not depend on each other, beside each other) and writes, per chunk, the entry state S, the exit-state
// gradient dS and dY; every other gradient is a product within one chunk, formed by the
// caller from these (dV = diag(beta) dY, the rest batched over chunks).
//
// MI355X mapping: one workgroup of kChainWaves waves per (chain, sequence-head, 16 kChainWaves
// state columns), each wave owning 16 columns (the recurrence never mixes V columns).
// The chunk's shared operands -- k rows, q rows, T (forward) or T^T (backward), Rq^T,
// 64 x 64 or 64 x d 16-bit tiles -- are staged in LDS with rows padded
// by 16 bytes (the 16-lane fragment reads then touch 16 distinct bank groups); k^T and q^T
// fragments come from the rows by transposing reads.  Products run on
// v_mfma_f32_16x16x32 (fp32 accumulation); the state and every per-column intermediate
// (Y, U, dU, dY) go through a per-wave transposed bf16 buffer ([column][k], 16 bytes per
// lane per fragment) to become the B operand of the next product.
// Bound by the latency of a chunk's chain of products and LDS exchanges, with one wave per
// SIMD: 8 sequences of 2,048 tokens, 8 heads, d = 128 take 167 us; 247 with one chain after the
// other on two of a CU's four SIMDs and with k^T, q^T and (diag(Ga) dO)^T read as tiles of their own.
#include <initializer_list>
#include <type_traits>

#include "common.h"

namespace atma {

// Per-token factor rows of a chunk: Ga, w, beta, Ga_C, lg, then the l2-norm factors of
// the q and k rows: iq = scale / max(|q|, eps), ik = 1 / max(|k|, eps) (scale and 1 without
// l2norm) and uq2 = 1 / |q|^2, uk2 = 1 / |k|^2 where the norm exceeds eps (else 0; 0
// without l2norm), all 0 past the sequence's end.
constexpr int kFRows = 9;

struct Bwd16ChainArgs {
  const void* kr;    // [N][64][D]  k rows of each chunk (N = BH * NC, chunk-head major)
  const void* qr;    // [N][64][D]  q rows (scaled, normalised)
  const void* tm;    // [N][64][64] T
  const void* tt;    // [N][64][64] T^T
  const void* rt;    // [N][64][64] Rq^T
  const void* vt;    // [N][D][64]  v^T
  const void* ot;    // [N][D][64]  dO^T
  const float* f;    // [N][5][64]  Ga, w, beta, Ga_C (all 64 entries), lg
  const float* s0;   // [BH][D][D] initial state, or null (zero)
  const float* dst;  // [BH][D][D] final-state cotangent, or null (zero)
  void* s_entry;     // [N][D][D]  out (16-bit): each chunk's entry state
  void* ds_end;      // [N][D][D]  out (16-bit): the gradient of each chunk's exit state
  void* u;           // [N][64][D] out (16-bit): U = T diag(beta) (V - diag(Ga) K S)
  float* dy;         // [N][64][D] out: dY
  float* ds0;        // [BH][D][D] out: the gradient of the initial state
  int BH, NC;
};

// LDS bytes of a chain workgroup: two of them share a CU, one per SIMD pair.
template <int D>
struct ChainLds {
  static constexpr int NW = 2, C = 64, PD = D + 8, PC = C + 8;  // padded pitches (elements)
  static constexpr int Kr = 0, Tm = Kr + 2 * C * PD, Fs = Tm + 2 * C * PC, Sb = Fs + 4 * 4 * C, X1 = Sb + NW * 32 * PD,
                       X2 = X1 + NW * 32 * PC, Fwd = X2 + NW * 32 * PC;
  static constexpr int Qr = Fwd, Rt = Qr + 2 * C * PD, XO = Rt + 2 * C * PC, Bwd = XO + NW * 32 * PC;
  static_assert(Bwd <= 80 * 1024, "two workgroups per CU");
};

// A contiguous 16-bit tile of N * NTH 16-byte chunks: thread tid (of NTH) holds chunks
// tid + NTH j.
template <int N, int NTH = 256>
__device__ __forceinline__ void tile_load(u32x4 (&r)[N], const void* src, int tid) {
  const u32x4* s = (const u32x4*)src;
#pragma unroll
  for (int j = 0; j < N; ++j) r[j] = s[tid + NTH * j];
}
// ... into LDS rows of CPR chunks, padded to PITCH elements
template <int N, int CPR, int PITCH, int NTH = 256, typename T>
__device__ __forceinline__ void tile_store(T* dst, const u32x4 (&r)[N], int tid) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = tid + NTH * j;
    *(u32x4*)(dst + (i / CPR) * PITCH + 8 * (i % CPR)) = r[j];
  }
}

// Waves (16 state columns each) per workgroup of the chain kernel: two, so that 64
// sequence-heads of d = 128 run 256 workgroups of each chain, one of both per CU.
constexpr int kChainWaves = 2;

template <typename T, int D>
__global__ void __launch_bounds__(64 * kChainWaves, 1) gdn_bwd16_chain_kernel(Bwd16ChainArgs a) {
  constexpr int NW = kChainWaves, NTH = 64 * NW, WC = 16 * NW;  // waves, threads, columns
  using L = ChainLds<D>;
  constexpr int C = 64, PD = L::PD, PC = L::PC;
  static_assert(L::NW == NW, "waves");
  constexpr int KS = D / 32;                      // 32-wide k steps over D
  constexpr int DT = D / 16;                      // 16-row tiles over D
  static_assert(D % WC == 0 && 4 * C % NTH == 0, "whole column slabs and factor rows");
  __shared__ __attribute__((aligned(16))) char lds[L::Bwd];
  T* Kr = (T*)(lds + L::Kr);
  T* Qr = (T*)(lds + L::Qr);
  T* Tm = (T*)(lds + L::Tm);  // T in the forward chain, T^T in the backward
  T* Rt = (T*)(lds + L::Rt);
  float* Fs = (float*)(lds + L::Fs);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  T* Sb = (T*)(lds + L::Sb) + wave * 16 * PD;  // S^T / dS^T of the wave's columns
  T* X1 = (T*)(lds + L::X1) + wave * 16 * PC;
  T* X2 = (T*)(lds + L::X2) + wave * 16 * PC;
  T* XO = (T*)(lds + L::XO) + wave * 16 * PC;  // dO^T rows of the wave's columns
  // the forward chains first, then the backward ones; the column slabs of one sequence-head
  // go to one XCD (workgroup i runs on XCD i % 8), whose L2 then serves its tiles
  constexpr int SL = D / WC;
  const int nwg = a.BH * SL;
  const bool fwd = (int)blockIdx.x < nwg;
  const int wg = fwd ? blockIdx.x : blockIdx.x - nwg;
  int bh = wg / SL, slab = wg % SL;
  if (a.BH % 8 == 0) {
    bh = (wg >> 3) / SL * 8 + (wg & 7);
    slab = (wg >> 3) % SL;
  }
  const int v0 = WC * slab + 16 * wave;  // the wave's first column
  const int col = v0 + c16;                                  // the lane's column (C layout)

  constexpr int NT = C * D / 8 / NTH;   // chunks per thread of a 64 x D or D x 64 tile
  constexpr int NTM = C * C / 8 / NTH;  // ... of a 64 x 64 tile
  constexpr int NF = 4 * C / NTH;       // factor entries per thread
  // the wave's 16 rows of a [D][64] tile: 2 chunks per lane
  auto rows16_load = [&](u32x4 (&r)[2], const void* src) {
    const u32x4* s = (const u32x4*)src;
    r[0] = s[lane];
    r[1] = s[lane + 64];
  };
  auto rows16_store = [&](T* dst, const u32x4 (&r)[2]) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int i = lane + 64 * k;
      *(u32x4*)(dst + (i >> 3) * PC + 8 * (i & 7)) = r[k];
    }
  };
  // fragment: row (row0 + c16) of a padded tile, 8 elements from column k0 + 8 g (the A
  // operand of rows row0 .. + 15, or the B operand of 16 columns from a [column][k] buffer)
  auto frag = [&](const T* tile, int pitch, int row0, int k0) {
    return *(const u32x4*)(tile + (row0 + c16) * pitch + k0 + 8 * g);
  };
  // fragment of the transpose: rows col0 + [0, 16) are columns of a row tile, k its rows k0 + 8 g + [0, 8), by
  // transposing reads (lane s of a 16-lane group reads row + s / 4, columns 4 (s % 4) .., lane i gets column i)
  auto frag_t = [&](const T* tile, int col0, int k0) {
    const T* p = tile + (k0 + 8 * g + (c16 >> 2)) * PD + col0 + 4 * (c16 & 3);
    const u32x2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * PD);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  // C tile t (rows 16 t + 4 g + i, column c16) into a [column][row] buffer
  auto put_t = [&](T* buf, int pitch, int t, const f32x4& x) {
    const u32x2 pk = {pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3])};
    *(u32x2*)(buf + c16 * pitch + 16 * t + 4 * g) = pk;
  };
  auto rows_of = [&](int t, int i) { return 16 * t + 4 * g + i; };
  // the wave's [16 columns][K] 16-bit tile (pitch P) out as K rows of a [K][D] output at
  // columns v0 .. v0 + 15, by transposing reads: 16-byte stores of 8 columns of one row
  // instead of one 2-byte store per element
  auto store_cols = [&](const T* buf, int pitch, auto K_c, T* out) {
    constexpr int K = decltype(K_c)::value;
    const int q = lane >> 4, sl = lane & 15, rr = sl >> 2, cc = 4 * (sl & 3);
#pragma unroll
    for (int u = q; u < 2 * (K / 16); u += 4) {
      const int r0 = 8 * (u & 1), c0 = 16 * (u >> 1);
      const u32x2 lo = lds_read_tr16(buf + (r0 + rr) * pitch + c0 + cc);
      const u32x2 hi = lds_read_tr16(buf + (r0 + 4 + rr) * pitch + c0 + cc);
      *(u32x4*)(out + (int64_t)(c0 + sl) * D + v0 + r0) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };

  // ---------------------------------------------------------------- forward chain
  // the next chunk's operands are loaded into registers while this one computes
  u32x4 rk[NT], rtm[NTM];
  float rf[NF];
  if (fwd) {
    f32x4 S[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        S[t][i] = a.s0 ? a.s0[((int64_t)bh * D + rows_of(t, i)) * D + col] : 0.f;

    u32x2 rv[4];
    auto fwd_load = [&](int64_t n) {
      tile_load<NT, NTH>(rk, (const T*)a.kr + n * C * D, tid);
      tile_load<NTM, NTH>(rtm, (const T*)a.tm + n * C * C, tid);
#pragma unroll
      for (int j = 0; j < NF; ++j) rf[j] = a.f[n * kFRows * C + tid + NTH * j];
      const T* vrow = (const T*)a.vt + (n * D + col) * C;
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) rv[rt] = *(const u32x2*)(vrow + 16 * rt + 4 * g);
    };
    fwd_load((int64_t)bh * a.NC);
    for (int c = 0; c < a.NC; ++c) {
      const int64_t n = (int64_t)bh * a.NC + c;
      __syncthreads();  // every wave is done with the previous chunk's tiles
      tile_store<NT, D / 8, PD, NTH>(Kr, rk, tid);
      tile_store<NTM, 8, PC, NTH>(Tm, rtm, tid);
#pragma unroll
      for (int j = 0; j < NF; ++j) Fs[tid + NTH * j] = rf[j];
      f32x4 Vc[4];  // v of the lane's column, C layout (rows = tokens)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const u32x4 x = {rv[rt][0], rv[rt][1], 0, 0};
        Vc[rt] = f32x4{elem16<T>(x, 0), elem16<T>(x, 1), elem16<T>(x, 2), elem16<T>(x, 3)};
      }
      if (c + 1 < a.NC) fwd_load(n + 1);
#pragma unroll
      for (int t = 0; t < DT; ++t) put_t(Sb, PD, t, S[t]);
      __syncthreads();

      // Z = K S
      f32x4 Z[4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) Z[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4 bf = frag(Sb, PD, 0, 32 * s);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) Z[rt] = mfma16x16x32<T>(frag(Kr, PD, 16 * rt, 32 * s), bf, Z[rt]);
      }
      // Y = diag(beta) (V - diag(Ga) Z)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        f32x4 y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = rows_of(rt, i);
          y[i] = Fs[2 * C + p] * (Vc[rt][i] - Fs[p] * Z[rt][i]);
        }
        put_t(X1, PC, rt, y);
      }
      wave_sync();
      // U = T Y, then w U
      f32x4 U[4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) U[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4 bf = frag(X1, PC, 0, 32 * s);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) U[rt] = mfma16x16x32<T>(frag(Tm, PC, 16 * rt, 32 * s), bf, U[rt]);
      }
      // U out through the wave's X1 buffer (its Y^T operand reads are done: in order, one wave)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) put_t(X1, PC, rt, U[rt]);
      wave_sync();
      store_cols(X1, PC, std::integral_constant<int, C>{}, (T*)a.u + n * C * D);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = Fs[C + rows_of(rt, i)] * U[rt][i];
        put_t(X2, PC, rt, x);
      }
      wave_sync();
      // the entry state, then S <- Ga_C S + K^T diag(w) U
      store_cols(Sb, PD, std::integral_constant<int, D>{}, (T*)a.s_entry + n * D * D);  // S^T of this step
      const float gC = Fs[3 * C];
#pragma unroll
      for (int t = 0; t < DT; ++t) S[t] *= gC;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4 bf = frag(X2, PC, 0, 32 * s);
#pragma unroll
        for (int t = 0; t < DT; ++t) S[t] = mfma16x16x32<T>(frag_t(Kr, 16 * t, 32 * s), bf, S[t]);
      }
    }

    return;
  }

  // ---------------------------------------------------------------- backward chain
  f32x4 dS[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dS[t][i] = a.dst ? a.dst[((int64_t)bh * D + rows_of(t, i)) * D + col] : 0.f;

  u32x4 rq[NT], rrt[NTM], ro[2];
  auto bwd_load = [&](int64_t n) {
    tile_load<NT, NTH>(rk, (const T*)a.kr + n * C * D, tid);
    tile_load<NT, NTH>(rq, (const T*)a.qr + n * C * D, tid);
    tile_load<NTM, NTH>(rtm, (const T*)a.tt + n * C * C, tid);
    tile_load<NTM, NTH>(rrt, (const T*)a.rt + n * C * C, tid);
#pragma unroll
    for (int j = 0; j < NF; ++j) rf[j] = a.f[n * kFRows * C + tid + NTH * j];
    rows16_load(ro, (const T*)a.ot + (n * D + v0) * C);
  };
  bwd_load((int64_t)bh * a.NC + a.NC - 1);
  for (int c = a.NC - 1; c >= 0; --c) {
    const int64_t n = (int64_t)bh * a.NC + c;
    __syncthreads();
    tile_store<NT, D / 8, PD, NTH>(Kr, rk, tid);
    tile_store<NT, D / 8, PD, NTH>(Qr, rq, tid);
    tile_store<NTM, 8, PC, NTH>(Tm, rtm, tid);
    tile_store<NTM, 8, PC, NTH>(Rt, rrt, tid);
#pragma unroll
    for (int j = 0; j < NF; ++j) Fs[tid + NTH * j] = rf[j];
    rows16_store(XO, ro);
    if (c > 0) bwd_load(n - 1);
#pragma unroll
    for (int t = 0; t < DT; ++t) put_t(Sb, PD, t, dS[t]);
    __syncthreads();
    // the exit-state gradient of this chunk, from its 16-bit transpose
    store_cols(Sb, PD, std::integral_constant<int, D>{}, (T*)a.ds_end + n * D * D);

    // dU = diag(w) K dS + Rq^T dO
    f32x4 dU[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) dU[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4 bf = frag(Sb, PD, 0, 32 * s);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) dU[rt] = mfma16x16x32<T>(frag(Kr, PD, 16 * rt, 32 * s), bf, dU[rt]);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) dU[rt][i] *= Fs[C + rows_of(rt, i)];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const u32x4 bf = frag(XO, PC, 0, 32 * s);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) dU[rt] = mfma16x16x32<T>(frag(Rt, PC, 16 * rt, 32 * s), bf, dU[rt]);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) put_t(X1, PC, rt, dU[rt]);
    wave_sync();
    // dY = T^T dU
    f32x4 dY[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) dY[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const u32x4 bf = frag(X1, PC, 0, 32 * s);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) dY[rt] = mfma16x16x32<T>(frag(Tm, PC, 16 * rt, 32 * s), bf, dY[rt]);
    }
    float* dyo = a.dy + n * C * D;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = rows_of(rt, i);
        dyo[p * D + col] = dY[rt][i];
        x[i] = -Fs[p] * Fs[2 * C + p] * dY[rt][i];
      }
      put_t(X2, PC, rt, x);
    }
    wave_sync();
    // dS <- Ga_C dS + Q^T diag(Ga) dO - K^T diag(Ga beta) dY
    const float gC = Fs[3 * C];
#pragma unroll
    for (int t = 0; t < DT; ++t) dS[t] *= gC;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u32x4 b1 = frag(XO, PC, 0, 32 * s);  // diag(Ga) dO, rounded as a 16-bit operand
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float* ga = Fs + 32 * s + 8 * g + 2 * e;
        b1[e] = pack2<T>(ga[0] * elem16<T>(b1, 2 * e), ga[1] * elem16<T>(b1, 2 * e + 1));
      }
      const u32x4 b2 = frag(X2, PC, 0, 32 * s);
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        dS[t] = mfma16x16x32<T>(frag_t(Qr, 16 * t, 32 * s), b1, dS[t]);
        dS[t] = mfma16x16x32<T>(frag_t(Kr, 16 * t, 32 * s), b2, dS[t]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) a.ds0[((int64_t)bh * D + rows_of(t, i)) * D + col] = dS[t][i];
}

// ------------------------------------------------------------------------------ prep
// One workgroup per chunk-head item n (4 waves): the operand tiles of the chain and of the
// chunk-local gradients.  The raw k, q rows are l2-normalised (q also scaled, as the
// forward does: x / max(|x|, 1e-12)) and rounded to 16 bits once; wave P
// forms row block P of K K^T and Q K^T on MFMA and from them Rq^T and the 16 x 16 blocks of
// N = diag(beta) A (fp32, LDS); then wave 0 inverts I + N -- the four diagonal blocks by
// forward substitution (lane (g, c) solves column c of block g), the blocks below them by
// fp32 block products on v_mfma_f32_16x16x4f32 -- while waves 1-3 write the transposed
// tiles v^T and dO^T from the LDS rows by transposing reads;
// last, every wave writes T and T^T.
struct Bwd16PrepArgs {
  const void* q;      // (B, T, H, D) 16-bit, raw
  const void* dO;     // (B, T, H, D) 16-bit
  const void* k;      // (B, T, H / G, D) 16-bit, raw
  const void* v;      // (B, T, H / G, D) 16-bit
  const float* g;     // (B, T, H) log decay
  const float* beta;  // (B, T, H)
  void *kr, *qr, *tm, *tt, *rt, *vt, *ot;
  float* f;
  float scale;
  int l2norm;
  int B, T, H, NC, G;
};

// Sum over each group of 8 lanes (the two quads of each half row), in every lane.
__device__ __forceinline__ float row8_sum(float x) {
  x += dpp_f32<0xB1>(x);
  x += dpp_f32<0x4E>(x);
  return x + dpp_f32<0x141>(x);
}

// e^x on the hardware exp2 (about 1 ulp), for the prep's per-element decay factors
__device__ __forceinline__ float exp_hw(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

template <typename T, int D>
__global__ void __launch_bounds__(256) gdn_bwd16_prep_kernel(Bwd16PrepArgs a) {
  constexpr int C = 64, PD = D + 8, PT = C + 8, KS = D / 32;
  constexpr int NV = D / 32;  // 16-byte row chunks per thread
  __shared__ __attribute__((aligned(16))) T Ks[C * PD];
  __shared__ __attribute__((aligned(16))) T Qs[C * PD];
  __shared__ __attribute__((aligned(16))) T Vs[C * PD];
  __shared__ __attribute__((aligned(16))) T Os[C * PD];
  // N = diag(beta) A in 16 x 16 blocks: the diagonal blocks as N^T (rows of 16 floats, the
  // substitution's columns) and the six blocks below them in the transposed accumulator
  // layout the block products take (register i of lane (g, c) of block (S, P), S < P:
  // N[16P + c][16S + 4g + i]).  Only wave 0 reads them, in order, so the substitution's
  // T^T diagonal blocks (Mb) overwrite the N^T ones it has consumed, and T, row-major 16-bit,
  // overwrites all of it at the end (84 KiB in all would allow one workgroup per CU; 79 KiB
  // allows two, so one's loads overlap the other's products)
  __shared__ __attribute__((aligned(16))) float Nd[4 * 256 + 6 * 256];
  __shared__ float Lg[C], Bt[C];
  float* Mb = Nd;  // T^T of the diagonal blocks
  T* Tl = (T*)Nd;  // T, row-major, pitch PT
  static_assert(C * PT * (int)sizeof(T) <= (int)sizeof(Nd), "T fits the N blocks' bytes");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int64_t n = blockIdx.x;
  const int bh = (int)(n / a.NC), c = (int)(n % a.NC);
  const int b = bh / a.H, h = bh % a.H;
  const int rows = min(a.T - c * C, C);
  const int64_t tok0 = (int64_t)b * a.T + (int64_t)c * C;
  const int64_t rs = (int64_t)a.H * D, krs = (int64_t)(a.H / a.G) * D;  // token strides (elements)
  const int64_t base = tok0 * rs + (int64_t)h * D, kbase = tok0 * krs + (int64_t)(h / a.G) * D;

  // rows (zero past the sequence's end), all loads issued before the stores
  {
    u32x4 kx[NV], qx[NV], vx[NV], ox[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = tid + 256 * j, r = i / (D / 8), ch = i % (D / 8);
      kx[j] = qx[j] = vx[j] = ox[j] = u32x4{0u, 0u, 0u, 0u};
      if (r < rows) {
        const int64_t o = base + r * rs + 8 * ch, ok = kbase + r * krs + 8 * ch;
        kx[j] = *(const u32x4*)((const T*)a.k + ok);
        qx[j] = *(const u32x4*)((const T*)a.q + o);
        vx[j] = *(const u32x4*)((const T*)a.v + ok);
        ox[j] = *(const u32x4*)((const T*)a.dO + o);
      }
    }
    float gl = 0.f, bt = 0.f;
    if (wave == 0 && lane < rows) {
      gl = a.g[(tok0 + lane) * a.H + h];
      bt = a.beta[(tok0 + lane) * a.H + h];
    }
    float* fo = a.f + n * kFRows * C;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = tid + 256 * j, r = i / (D / 8), ch = i % (D / 8);
      // row norms: a row's D / 8 chunks sit in D / 8 consecutive lanes
      float sk = 0.f, sq = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // packed pairs (v_dot2)
        sk = dot2<T>(kx[j][e], kx[j][e], sk);
        sq = dot2<T>(qx[j][e], qx[j][e], sq);
      }
      if constexpr (D == 128) {
        sk = row16_sum(sk);
        sq = row16_sum(sq);
      } else {
        sk = row8_sum(sk);
        sq = row8_sum(sq);
      }
      const float nk = sqrtf(sk), nq = sqrtf(sq);
      const bool ok = r < rows;
      const float ik = !ok ? 0.f : a.l2norm ? __builtin_amdgcn_rcpf(fmaxf(nk, 1e-12f)) : 1.f;
      const float iq = !ok ? 0.f : (a.l2norm ? __builtin_amdgcn_rcpf(fmaxf(nq, 1e-12f)) : 1.f) * a.scale;
      if (ch == 0) {
        fo[5 * C + r] = iq;
        fo[6 * C + r] = ik;
        fo[7 * C + r] = ok && a.l2norm && nq > 1e-12f ? __builtin_amdgcn_rcpf(sq) : 0.f;
        fo[8 * C + r] = ok && a.l2norm && nk > 1e-12f ? __builtin_amdgcn_rcpf(sk) : 0.f;
      }
      u32x4 kp, qp;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kp[e] = pack2<T>(ik * elem16<T>(kx[j], 2 * e), ik * elem16<T>(kx[j], 2 * e + 1));
        qp[e] = pack2<T>(iq * elem16<T>(qx[j], 2 * e), iq * elem16<T>(qx[j], 2 * e + 1));
      }
      *(u32x4*)(Ks + r * PD + 8 * ch) = kp;
      *(u32x4*)(Qs + r * PD + 8 * ch) = qp;
      *(u32x4*)((T*)a.kr + (n * C + r) * D + 8 * ch) = kp;
      *(u32x4*)((T*)a.qr + (n * C + r) * D + 8 * ch) = qp;
      *(u32x4*)(Vs + r * PD + 8 * ch) = vx[j];
      *(u32x4*)(Os + r * PD + 8 * ch) = ox[j];
    }
    if (wave == 0) {  // inclusive prefix sum of the log decays, per-token factors
      float lg = gl;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(lg, off, 64);
        if (lane >= off) lg += y;
      }
      const float lgC = __shfl(lg, 63, 64);
      const float ga = exp_hw(lg);
      Lg[lane] = lg;
      Bt[lane] = bt;
      fo[lane] = ga;
      fo[C + lane] = exp_hw(lgC - lg);
      fo[2 * C + lane] = bt;
      fo[3 * C + lane] = exp_hw(lgC);
      fo[4 * C + lane] = lg;
    }
  }
  __syncthreads();

  // row block P = wave of K K^T and Q K^T: Rq^T, the diagonal N block and, from the blocks
  // right of the diagonal (Gram symmetry), the N blocks below it in the block products' layout
  {
    const int P = wave;
    u32x4 ka[KS], qa[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      ka[s] = *(const u32x4*)(Ks + (16 * P + c16) * PD + 32 * s + 8 * g);
      qa[s] = *(const u32x4*)(Qs + (16 * P + c16) * PD + 32 * s + 8 * g);
    }
#pragma unroll
    for (int S = 0; S < 4; ++S) {
      f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4 kb = *(const u32x4*)(Ks + (16 * S + c16) * PD + 32 * s + 8 * g);
        kk = mfma16x16x32<T>(ka[s], kb, kk);
        qk = mfma16x16x32<T>(qa[s], kb, qk);
      }
      // lane (g, c16) register i: token pair (16 P + 4g + i, 16 S + c16)
      const int sc = 16 * S + c16;
      const float lgs = Lg[sc];
      f32x4 rq;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = 16 * P + 4 * g + i;
        rq[i] = sc <= p ? exp_hw(Lg[p] - lgs) * qk[i] : 0.f;
      }
      *(u32x2*)((T*)a.rt + (n * C + sc) * C + 16 * P + 4 * g) = u32x2{pack2<T>(rq[0], rq[1]), pack2<T>(rq[2], rq[3])};
      if (S == P) {  // N^T[c][4g + i] = N[16P + 4g + i][16P + c], strictly lower
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = 16 * P + 4 * g + i;
          v[i] = c16 < 4 * g + i ? Bt[p] * exp_hw(Lg[p] - lgs) * kk[i] : 0.f;
        }
        *(f32x4*)(Nd + P * 256 + c16 * 16 + 4 * g) = v;
      } else if (S > P) {  // N[16S + c][16P + 4g + i] = beta_r e^(lg_r - lg_s) k_s . k_r
        const int r = sc;
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = Bt[r] * exp_hw(Lg[r] - Lg[16 * P + 4 * g + i]) * kk[i];
        *(f32x4*)(Nd + 4 * 256 + tri(P, S - 1) * 256 + lane * 4) = v;
      }
    }
  }
  __syncthreads();

  if (wave == 0) {
    // T = (I + N)^-1.  The diagonal blocks by forward substitution in fp32: lane (g, c) solves
    // column c of block g, N^T rows read from LDS
    {
      const float* nt = Nd + g * 256;
      float x[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = (r == c16) ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < 15; ++j) {
        float nv[16];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const f32x4 v = *(const f32x4*)(nt + j * 16 + 4 * q4);  // column j of N
#pragma unroll
          for (int e = 0; e < 4; ++e) nv[4 * q4 + e] = v[e];
        }
#pragma unroll
        for (int r = j + 1; r < 16; ++r) x[r] = fmaf(-nv[r], x[j], x[r]);
      }
      float* mt = Mb + g * 256 + c16 * 16;  // T^T row c = column c of T
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) *(f32x4*)(mt + 4 * q4) = f32x4{x[4 * q4], x[4 * q4 + 1], x[4 * q4 + 2], x[4 * q4 + 3]};
    }
    wave_sync();
    f32x4 tpp[4], tppT[4], at[6];  // T_PP and T_PP^T in the accumulator layout
#pragma unroll
    for (int P = 0; P < 4; ++P) {
      tpp[P] = *(const f32x4*)(Mb + P * 256 + c16 * 16 + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) tppT[P][i] = Mb[P * 256 + (4 * g + i) * 16 + c16];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) at[k] = *(const f32x4*)(Nd + 4 * 256 + k * 256 + lane * 4);
    // off-diagonal blocks, level L = P - S: T_PS = -T_PP Y_PS with Y_PS = sum_{k=S}^{P-1}
    // N_Pk T_kS, and (T^T)_SP = -Y_PS^T T_PP^T (at(k, P) = block (k, P) of the layout above)
    auto atb = [&](int k, int P) { return at[tri(k, P - 1)]; };
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    const f32x4 y10 = blk_mul(atb(0, 1), tpp[0], z);
    const f32x4 y21 = blk_mul(atb(1, 2), tpp[1], z);
    const f32x4 y32 = blk_mul(atb(2, 3), tpp[2], z);
    const f32x4 t10 = -blk_mul(tppT[1], y10, z);
    const f32x4 t21 = -blk_mul(tppT[2], y21, z);
    const f32x4 tt01 = -blk_mul(y10, tppT[1], z);
    const f32x4 tt12 = -blk_mul(y21, tppT[2], z);
    const f32x4 tt23 = -blk_mul(y32, tppT[3], z);
    const f32x4 y20 = blk_mul(atb(1, 2), t10, blk_mul(atb(0, 2), tpp[0], z));
    const f32x4 y31 = blk_mul(atb(2, 3), t21, blk_mul(atb(1, 3), tpp[1], z));
    const f32x4 t20 = -blk_mul(tppT[2], y20, z);
    const f32x4 tt02 = -blk_mul(y20, tppT[2], z);
    const f32x4 tt13 = -blk_mul(y31, tppT[3], z);
    const f32x4 y30 = blk_mul(atb(2, 3), t20, blk_mul(atb(1, 3), t10, blk_mul(atb(0, 3), tpp[0], z)));
    const f32x4 tt03 = -blk_mul(y30, tppT[3], z);
    // T row-major in 16 bits over the N blocks (every read of them is above): the T^T-form
    // block (S, P) gives row 16P + c, columns 16S + 4g .. + 3 of T (zeros above the diagonal)
    const f32x4 tb[4][4] = {{tppT[0], z, z, z}, {tt01, tppT[1], z, z}, {tt02, tt12, tppT[2], z},
                            {tt03, tt13, tt23, tppT[3]}};
#pragma unroll
    for (int P = 0; P < 4; ++P)
#pragma unroll
      for (int S = 0; S < 4; ++S) {
        const f32x4 v = tb[P][S];
        *(u32x2*)(Tl + (16 * P + c16) * PT + 16 * S + 4 * g) = u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
      }
  } else {
    // [D][64] tiles from the LDS rows by transposing reads: a 16-lane group reads 8 rows x 16
    // columns (lane s: row r0 + s / 4 (+ 4), columns c0 + 4 (s % 4) ..), lane i then holds
    // tokens r0 .. r0 + 7 of column c0 + i, one 16-byte chunk of row d = c0 + i of the tile
    const int gi = (tid - 64) >> 4, sl = lane & 15;  // 12 groups of 16 lanes
    const int rr = sl >> 2, cc = 4 * (sl & 3);
    constexpr int UNITS = 2 * (D / 16) * 8;          // (tile, 16-column block, 8-row block)
    for (int u = gi; u < UNITS; u += 12) {
      const int tile = u / ((D / 16) * 8), rem = u % ((D / 16) * 8);
      const int c0 = 16 * (rem / 8), r0 = 8 * (rem % 8);
      const T* src = tile == 0 ? Vs : Os;
      const u32x2 lo = lds_read_tr16(src + (r0 + rr) * PD + c0 + cc);
      const u32x2 hi = lds_read_tr16(src + (r0 + 4 + rr) * PD + c0 + cc);
      *(u32x4*)((T*)(tile == 0 ? a.vt : a.ot) + (n * D + c0 + sl) * C + r0) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  }
  __syncthreads();
  // T and T^T out: 64 rows of 128 bytes each, two 16-byte chunks per thread
  {
    const int row = tid >> 2, ch = 2 * (tid & 3);  // ... chunks ch, ch + 1 of T's row
    T* tmo = (T*)a.tm + (n * C + row) * C;
#pragma unroll
    for (int k = 0; k < 2; ++k) *(u32x4*)(tmo + 8 * (ch + k)) = *(const u32x4*)(Tl + row * PT + 8 * (ch + k));
    // T^T by transposing reads: group gi (16 lanes) takes 16-column block c0 and two 8-row
    // blocks of T
    const int gi = tid >> 4, sl = lane & 15, rr = sl >> 2, cc = 4 * (sl & 3);
    const int c0 = 16 * (gi & 3);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r0 = 8 * (2 * (gi >> 2) + k);
      const u32x2 lo = lds_read_tr16(Tl + (r0 + rr) * PT + c0 + cc);
      const u32x2 hi = lds_read_tr16(Tl + (r0 + 4 + rr) * PT + c0 + cc);
      *(u32x4*)((T*)a.tt + (n * C + c0 + sl) * C + r0) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  }
}

// ------------------------------------------------------------------------------ local
// One workgroup per chunk-head item n (4 waves); wave w owns tokens 16 w .. 16 w + 15.
// Products on v_mfma_f32_16x16x32 (16-bit operands, fp32 accumulation): K K^T, Q K^T,
// dY U^T, dO U^T (64 x 64) give the weights GA, GR; then, transposed (rows = d, columns = the
// wave's tokens, so that a lane holds four consecutive d of one token),
// dK = (GA + GA^T) K + GR^T Q - diag(Ga beta) dY S0^T + diag(w) U dS^T
// and dQ = GR K + diag(Ga) dO S0^T.  The sums over d that the gradients of beta and the
// log decays take reduce to row sums of these products with k and q:
// rowsum(dY o K S0) = rowsum(K o dY S0^T), rowsum(dO o Q S0) = rowsum(Q o dO S0^T),
// rowsum(K dS o U) = rowsum(K o U dS^T).
// The k and q rows are normalised and rounded from the raw ones as the prep does (the raw
// ones are needed for the l2 norm's backward anyway).  LDS: k rows, GA^T and GR^T (their
// transposes, like those of the rows, by transposing reads), and two row tiles that hold U and q
// first and the entry state S0, then the exit-state gradient dS, afterwards: 75 KiB and at most 256
// registers, so two workgroups share a CU and one's loads pass under the other's products.
// Bound by memory: an item reads 192 KiB and writes 49 at d = 128.  8 sequences of 2,048
// tokens, 8 heads: 123 us; 249 with one workgroup per CU (147 KiB of LDS: each transpose a tile
// of its own, S0 and dS beside the rest), k^T and q^T read from memory and 2-byte accesses to
// the raw rows and the outputs.
struct Bwd16LocalArgs {
  const void *q, *dO;  // (B, T, H, D) 16-bit (q raw)
  const void *k, *v;   // (B, T, H / G, D) 16-bit (k raw)
  const float* f;      // [N][kFRows][64]
  const void *s_entry, *ds_end, *u;
  const float* dy;
  void *dq, *dk, *dv;  // (B, T, H, D) 16-bit
  float *dg, *db;      // (B, T, H)
  int B, T, H, NC, G;
};

template <typename T, int D>
__global__ void __launch_bounds__(256, 2) gdn_bwd16_local_kernel(Bwd16LocalArgs a) {
  constexpr int C = 64, PD = D + 8, PC = C + 8, KS = D / 32, DT = D / 16, NT = D / 32, NSS = D * D / 2048;
  __shared__ __attribute__((aligned(16))) T Kr[C * PD];
  __shared__ __attribute__((aligned(16))) T SS[2 * C * PD];  // U and q rows, then S0 rows, then dS rows
  __shared__ __attribute__((aligned(16))) T GAt[C * PC];     // GA^T
  __shared__ __attribute__((aligned(16))) T GRt[C * PC];     // GR^T
  __shared__ float Fs[kFRows * C];
  __shared__ float colp[4][C];
  __shared__ float dyv[C], dbv[C], dlgs[C], red[2][4];
  T* Us = SS;
  T* Qr = SS + C * PD;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int64_t n = blockIdx.x;
  const int bh = (int)(n / a.NC), c = (int)(n % a.NC);
  const int b = bh / a.H, h = bh % a.H;
  const int rows = min(a.T - c * C, C);
  const int64_t tok0 = (int64_t)b * a.T + (int64_t)c * C;
  const int64_t rs = (int64_t)a.H * D, krs = (int64_t)(a.H / a.G) * D;  // token strides
  const int64_t base = tok0 * rs + (int64_t)h * D, kbase = tok0 * krs + (int64_t)(h / a.G) * D;
  const int ra = 16 * wave + c16;  // the lane's token
  const float* fn = a.f + n * kFRows * C;

  // fragment of rows row0 .. of a row tile; of its transpose (rows col0 .., k = the tile's rows k0 + 8 g ..)
  auto frag = [&](const T* tile, int pitch, int row0, int k0) {
    return *(const u32x4*)(tile + (row0 + c16) * pitch + k0 + 8 * g);
  };
  auto frag_t = [&](const T* tile, int pitch, int col0, int k0) {
    const T* p = tile + (k0 + 8 * g + (c16 >> 2)) * pitch + col0 + 4 * (c16 & 3);
    const u32x2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * pitch);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };

  // ---- k, q (normalised, rounded) and U rows into LDS; the wave's dY, dO and v rows
  u32x4 doA[KS], dyA[KS], kA[KS], qA[KS];
  {
    u32x4 rk[NT], rq[NT], ru[NT], vA[KS];
    float fk[NT], fq[NT];
    tile_load(ru, (const T*)a.u + n * C * D, tid);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int i = tid + 256 * j, r = i / (D / 8), ch = i % (D / 8);
      rk[j] = rq[j] = u32x4{0u, 0u, 0u, 0u};
      if (r < rows) {
        rk[j] = *(const u32x4*)((const T*)a.k + kbase + r * krs + 8 * ch);
        rq[j] = *(const u32x4*)((const T*)a.q + base + r * rs + 8 * ch);
      }
      fq[j] = fn[5 * C + r];
      fk[j] = fn[6 * C + r];
    }
    f32x4 dyl[KS][2];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float* yr = a.dy + (n * C + ra) * D + 32 * s + 8 * g;
      dyl[s][0] = *(const f32x4*)yr;
      dyl[s][1] = *(const f32x4*)(yr + 4);
      doA[s] = vA[s] = u32x4{0u, 0u, 0u, 0u};
      if (ra < rows) {
        doA[s] = *(const u32x4*)((const T*)a.dO + base + ra * rs + 32 * s + 8 * g);
        vA[s] = *(const u32x4*)((const T*)a.v + kbase + ra * krs + 32 * s + 8 * g);
      }
    }
    const float bt = fn[2 * C + ra];
    for (int i = tid; i < kFRows * C; i += 256) Fs[i] = fn[i];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int i = tid + 256 * j, r = i / (D / 8), ch = i % (D / 8);
      u32x4 kp, qp;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kp[e] = pack2<T>(fk[j] * elem16<T>(rk[j], 2 * e), fk[j] * elem16<T>(rk[j], 2 * e + 1));
        qp[e] = pack2<T>(fq[j] * elem16<T>(rq[j], 2 * e), fq[j] * elem16<T>(rq[j], 2 * e + 1));
      }
      *(u32x4*)(Kr + r * PD + 8 * ch) = kp;
      *(u32x4*)(Qr + r * PD + 8 * ch) = qp;
    }
    tile_store<NT, D / 8, PD>(Us, ru, tid);
    // dV = diag(beta) dY and rowsum(dY o V) from the wave's rows; dY as an operand
    float part = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const f32x4 y0 = dyl[s][0], y1 = dyl[s][1];
      dyA[s] = u32x4{pack2<T>(y0[0], y0[1]), pack2<T>(y0[2], y0[3]), pack2<T>(y1[0], y1[1]), pack2<T>(y1[2], y1[3])};
#pragma unroll
      for (int e = 0; e < 4; ++e) part = fmaf(y0[e], elem16<T>(vA[s], e), fmaf(y1[e], elem16<T>(vA[s], 4 + e), part));
      if (ra < rows)
        *(u32x4*)((T*)a.dv + base + ra * rs + 32 * s + 8 * g) =
            u32x4{pack2<T>(bt * y0[0], bt * y0[1]), pack2<T>(bt * y0[2], bt * y0[3]),
                  pack2<T>(bt * y1[0], bt * y1[1]), pack2<T>(bt * y1[2], bt * y1[3])};
    }
    part += __shfl_xor(part, 16, 64);
    part += __shfl_xor(part, 32, 64);
    if (g == 0) dyv[ra] = part;
  }
  const float* Bf = Fs + 2 * C;
  const float* Lgf = Fs + 4 * C;
  u32x4 rss[NSS];  // S0, stored to LDS once U and q are done with
  tile_load(rss, (const T*)a.s_entry + n * D * D, tid);
  __syncthreads();
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kA[s] = frag(Kr, PD, 16 * wave, 32 * s);
    qA[s] = frag(Qr, PD, 16 * wave, 32 * s);
  }

  // ---- 64 x 64 products of the wave's rows: A, Rq, dL, dRq, and the weights GA, GR
  {
    float dbl[4] = {0.f, 0.f, 0.f, 0.f}, lgl[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int S = 0; S < 4; ++S) {
      f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = kk, yl = kk, ou = kk;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4 kb = frag(Kr, PD, 16 * S, 32 * s), ub = frag(Us, PD, 16 * S, 32 * s);
        kk = mfma16x16x32<T>(kA[s], kb, kk);
        qk = mfma16x16x32<T>(qA[s], kb, qk);
        yl = mfma16x16x32<T>(dyA[s], ub, yl);
        ou = mfma16x16x32<T>(doA[s], ub, ou);
      }
      const int sc = 16 * S + c16, p0 = 16 * wave + 4 * g;
      const float lgs = Lgf[sc];
      f32x4 ga, gr;
      float colv = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = p0 + i;
        const float e = sc <= p ? exp_hw(Lgf[p] - lgs) : 0.f;
        const float A = sc < p ? e * kk[i] : 0.f;
        const float Rq = e * qk[i];
        const float dL = sc < p ? -yl[i] : 0.f;
        const float dA = Bf[p] * dL;
        const float dRq = sc <= p ? ou[i] : 0.f;
        ga[i] = dA * e;
        gr[i] = dRq * e;
        dbl[i] = fmaf(dL, A, dbl[i]);
        const float x = fmaf(dA, A, dRq * Rq);
        lgl[i] += x;
        colv += x;
      }
      *(u32x2*)(GAt + sc * PC + p0) = u32x2{pack2<T>(ga[0], ga[1]), pack2<T>(ga[2], ga[3])};
      *(u32x2*)(GRt + sc * PC + p0) = u32x2{pack2<T>(gr[0], gr[1]), pack2<T>(gr[2], gr[3])};
      colv += __shfl_xor(colv, 16, 64);
      colv += __shfl_xor(colv, 32, 64);
      if (g == 0) colp[wave][sc] = colv;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = row16_sum(dbl[i]), y = row16_sum(lgl[i]);
      if (c16 == 0) {
        dbv[16 * wave + 4 * g + i] = x;
        dlgs[16 * wave + 4 * g + i] = y;
      }
    }
  }
  __syncthreads();

  // ---- (GA + GA^T) K + GR^T Q and GR K, transposed: register i of tile t is d = 16 t + 4 g + i of token ra
  f32x4 dKn[DT], dQs[DT];
  {
    u32x4 g1[2], grt[2], gr[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const u32x4 mt = frag(GAt, PC, 16 * wave, 32 * j), m = frag_t(GAt, PC, 16 * wave, 32 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        g1[j][e] = pack2<T>(elem16<T>(m, 2 * e) + elem16<T>(mt, 2 * e), elem16<T>(m, 2 * e + 1) + elem16<T>(mt, 2 * e + 1));
      grt[j] = frag(GRt, PC, 16 * wave, 32 * j);
      gr[j] = frag_t(GRt, PC, 16 * wave, 32 * j);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      dKn[t] = dQs[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const u32x4 kb = frag_t(Kr, PD, 16 * t, 32 * j), qb = frag_t(Qr, PD, 16 * t, 32 * j);
        dKn[t] = mfma16x16x32<T>(kb, g1[j], dKn[t]);
        dKn[t] = mfma16x16x32<T>(qb, grt[j], dKn[t]);
        dQs[t] = mfma16x16x32<T>(kb, gr[j], dQs[t]);
      }
    }
  }
  __syncthreads();  // U and q are done with
  tile_store<NSS, D / 8, PD>(SS, rss, tid);
  u32x4 rds[NSS];
  tile_load(rds, (const T*)a.ds_end + n * D * D, tid);
  // the token's raw k and q (the lane's d): their rounded normalised rows for the row sums, the l2 norm's backward
  u32x2 kraw[DT], qraw[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    kraw[t] = qraw[t] = u32x2{0u, 0u};
    if (ra < rows) {
      kraw[t] = *(const u32x2*)((const T*)a.k + kbase + ra * krs + 16 * t + 4 * g);
      qraw[t] = *(const u32x2*)((const T*)a.q + base + ra * rs + 16 * t + 4 * g);
    }
  }
  const float Ga = Fs[ra], Wf = Fs[C + ra], Bt = Bf[ra], iq = Fs[5 * C + ra], ik = Fs[6 * C + ra];
  auto raw = [&](const u32x2& x, int i) { return elem16<T>(u32x4{x[0], x[1], 0u, 0u}, i); };
  auto unit = [&](float f, const u32x2& x, int i) {  // as rounded into the row tiles
    return elem16<T>(u32x4{pack2<T>(f * raw(x, i & ~1), f * raw(x, i | 1)), 0u, 0u, 0u}, i & 1);
  };
  __syncthreads();

  // ---- dY S0^T and dO S0^T, transposed
  float k1 = 0.f, q2 = 0.f, k3 = 0.f, xk = 0.f, xq = 0.f;
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    f32x4 P1 = {0.f, 0.f, 0.f, 0.f}, P2 = P1;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4 sb = frag(SS, PD, 16 * t, 32 * s);
      P1 = mfma16x16x32<T>(sb, dyA[s], P1);
      P2 = mfma16x16x32<T>(sb, doA[s], P2);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      k1 = fmaf(unit(ik, kraw[t], i), P1[i], k1);
      q2 = fmaf(unit(iq, qraw[t], i), P2[i], q2);
      dKn[t][i] -= Ga * Bt * P1[i];
      dQs[t][i] = fmaf(Ga, P2[i], dQs[t][i]);
      xq = fmaf(raw(qraw[t], i), dQs[t][i], xq);
    }
  }
  u32x4 uA[KS];  // (read again here: held from the start, they would not fit the registers)
#pragma unroll
  for (int s = 0; s < KS; ++s) uA[s] = *(const u32x4*)((const T*)a.u + (n * C + ra) * D + 32 * s + 8 * g);
  // <dS, S0> over the thread's chunks, then dS replaces S0
  {
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < NSS; ++j) {
      const int i = tid + 256 * j;
      const u32x4 sx = *(const u32x4*)(SS + (i / (D / 8)) * PD + 8 * (i % (D / 8)));
#pragma unroll
      for (int e = 0; e < 8; ++e) part = fmaf(elem16<T>(sx, e), elem16<T>(rds[j], e), part);
    }
    part = wave_sum(part);
    if (lane == 0) red[0][wave] = part;
  }
  __syncthreads();
  tile_store<NSS, D / 8, PD>(SS, rds, tid);
  __syncthreads();

  // ---- U dS^T, transposed
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    f32x4 P3 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) P3 = mfma16x16x32<T>(frag(SS, PD, 16 * t, 32 * s), uA[s], P3);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      k3 = fmaf(unit(ik, kraw[t], i), P3[i], k3);
      dKn[t][i] = fmaf(Wf, P3[i], dKn[t][i]);
      xk = fmaf(raw(kraw[t], i), dKn[t][i], xk);
    }
  }
  // sums over d: the lane's, then the four lanes of the token
  auto tok_sum = [&](float x) {
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
  };
  k1 = tok_sum(k1);
  q2 = tok_sum(q2);
  k3 = tok_sum(k3);
  // the l2 norm's backward: dx = i_x dX - i_x u_x2 x (x . dX) with x the raw row
  const float pq = iq * Fs[7 * C + ra] * tok_sum(xq), pk = ik * Fs[8 * C + ra] * tok_sum(xk);
  if (ra < rows) {
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      float x[4], y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = ik * dKn[t][i] - pk * raw(kraw[t], i);
        y[i] = iq * dQs[t][i] - pq * raw(qraw[t], i);
      }
      const int64_t o = base + ra * rs + 16 * t + 4 * g;
      *(u32x2*)((T*)a.dk + o) = u32x2{pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3])};
      *(u32x2*)((T*)a.dq + o) = u32x2{pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])};
    }
  }
  // gradients of beta and of the log decays
  if (g == 0) {
    if (ra < rows) a.db[(tok0 + ra) * a.H + h] = dyv[ra] - Ga * k1 + dbv[ra];
    dlgs[ra] += Ga * (q2 - Bt * k1) - Wf * k3;
  }
  const float wsum = wave_sum(g == 0 ? Wf * k3 : 0.f);
  if (lane == 0) red[1][wave] = wsum;
  __syncthreads();
  if (wave == 0) {
    float x = dlgs[lane] - (colp[0][lane] + colp[1][lane] + colp[2][lane] + colp[3][lane]);
    if (lane == C - 1)
      x += red[1][0] + red[1][1] + red[1][2] + red[1][3] +
           Fs[3 * C] * (red[0][0] + red[0][1] + red[0][2] + red[0][3]);
    // reverse cumulative sum: dg[p] = sum over s >= p
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float y = __shfl_down(x, off, 64);
      if (lane + off < 64) x += y;
    }
    if (lane < rows) a.dg[(tok0 + lane) * a.H + h] = x;
  }
}

// dk and dv summed over the G query heads of a group: out[row, hk] = sum_g in[row, hk G + g], rows of D 16-bit elements,
// fp32 accumulation, 8 elements per thread.  Bound by memory (8 x 2,048 tokens, 8 heads in groups of 4, d = 128, dk and dv:
// 84 MB in 15 us; one reduction each by torch 25, after expanded copies of k and v in 54).
template <typename T>
__global__ void __launch_bounds__(256) gdn_bwd16_group_sum_kernel(const u32x4* dk, const u32x4* dv, u32x4* dk_out,
                                                                  u32x4* dv_out, int64_t n, int G, int cpr) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // 16-byte chunk of the output, cpr per row
  if (i >= n) return;
  const u32x4* p = (blockIdx.y ? dv : dk) + i / cpr * G * cpr + i % cpr;
  float acc[8] = {};
  for (int g = 0; g < G; ++g) {
    const u32x4 x = p[(int64_t)g * cpr];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += elem16<T>(x, e);
  }
  (blockIdx.y ? dv_out : dk_out)[i] =
      u32x4{pack2<T>(acc[0], acc[1]), pack2<T>(acc[2], acc[3]), pack2<T>(acc[4], acc[5]), pack2<T>(acc[6], acc[7])};
}

}  // namespace atma

// ------------------------------------------------------------------------------ C ABI
namespace {

bool bwd16_dims_ok(int64_t d, int dtype, const char* who) {
  using namespace atma;
  if (d != 64 && d != 128) {
    set_error(ATMA_ERR_UNSUPPORTED, "%s: d = %lld (supported: 64, 128)", who, (long long)d);
    return false;
  }
  if (dtype != ATMA_BF16 && dtype != ATMA_F16) {
    set_error(ATMA_ERR_UNSUPPORTED, "%s: 16-bit operands only", who);
    return false;
  }
  return true;
}

bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if ((uintptr_t)p % 16) return false;
  return true;
}

}  // namespace

#define ATMA_BWD16_DISPATCH_NT(KERNEL, grid, nthreads, stream, args)                          \
  do {                                                                                        \
    if (dtype == ATMA_BF16) {                                                                 \
      if (d == 128) atma::KERNEL<atma::bf16, 128><<<grid, dim3(nthreads), 0, stream>>>(args); \
      else atma::KERNEL<atma::bf16, 64><<<grid, dim3(nthreads), 0, stream>>>(args);           \
    } else {                                                                                  \
      if (d == 128) atma::KERNEL<atma::f16, 128><<<grid, dim3(nthreads), 0, stream>>>(args);  \
      else atma::KERNEL<atma::f16, 64><<<grid, dim3(nthreads), 0, stream>>>(args);            \
    }                                                                                         \
  } while (0)
#define ATMA_BWD16_DISPATCH(KERNEL, grid, stream, args) ATMA_BWD16_DISPATCH_NT(KERNEL, grid, 256, stream, args)

extern "C" int atma_gated_delta_bwd16_prep(const void* q, const void* k, const void* v, const void* d_out,
                                           const float* g, const float* beta, void* kr, void* qr, void* tm, void* tt,
                                           void* rt, void* vt, void* ot, float* f, int64_t B, int64_t T, int64_t H,
                                           int64_t Hkv, int64_t d, float scale, int l2norm, int dtype, void* stream) {
  using namespace atma;
  if (!bwd16_dims_ok(d, dtype, "gated_delta_bwd16_prep")) return ATMA_ERR_UNSUPPORTED;
  if (B < 0 || T < 0 || H <= 0 || Hkv <= 0 || H % Hkv) return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_prep: bad sizes");
  const int64_t NC = (T + 63) / 64;
  if (B == 0 || NC == 0) return ATMA_OK;
  if (!q || !k || !v || !d_out || !g || !beta || !kr || !qr || !tm || !tt || !rt || !vt || !ot || !f)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_prep: null pointer");
  if (!aligned16({q, k, v, d_out, kr, qr, tm, tt, rt, vt, ot}))
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_prep: operands must be 16-byte aligned");
  if (B * H * NC > 0x7fffffff || B * T > 0x7fffffff)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_prep: sizes too large");
  Bwd16PrepArgs a{q, d_out, k, v, g, beta, kr, qr, tm, tt, rt, vt, ot, f, scale, l2norm ? 1 : 0,
                  (int)B, (int)T, (int)H, (int)NC, (int)(H / Hkv)};
  const dim3 grid((unsigned)(B * H * NC));
  ATMA_BWD16_DISPATCH(gdn_bwd16_prep_kernel, grid, (hipStream_t)stream, a);
  return check_launch("gated_delta_bwd16_prep");
}

extern "C" int atma_gated_delta_bwd16_chain(const void* kr, const void* qr, const void* tm, const void* tt,
                                            const void* rt, const void* vt, const void* ot, const float* f, const float* s0, const float* dst,
                                            void* s_entry, void* ds_end, void* u, float* dy, float* ds0,
                                            int64_t BH, int64_t NC, int64_t d, int dtype, void* stream) {
  using namespace atma;
  if (!bwd16_dims_ok(d, dtype, "gated_delta_bwd16_chain")) return ATMA_ERR_UNSUPPORTED;
  if (BH < 0 || NC < 0) return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_chain: bad sizes");
  if (BH == 0 || NC == 0) return ATMA_OK;
  if (!kr || !qr || !tm || !tt || !rt || !vt || !ot || !f || !s_entry || !ds_end || !u || !dy ||
      !ds0)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_chain: null pointer");
  if (!aligned16({kr, qr, tm, tt, rt, vt, ot, s_entry, ds_end, u, dy}))
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_chain: tiles and outputs must be 16-byte aligned");
  const int64_t slabs = d / (16 * kChainWaves);  // column slabs (workgroups) per sequence-head
  if (2 * BH * slabs > 0x7fffffff || BH * NC > 0x7fffffff)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_chain: sizes too large");
  Bwd16ChainArgs a{kr, qr, tm, tt, rt, vt, ot, f, s0, dst, s_entry, ds_end, u, dy, ds0,
                   (int)BH, (int)NC};
  const dim3 grid((unsigned)(2 * BH * slabs));
  ATMA_BWD16_DISPATCH_NT(gdn_bwd16_chain_kernel, grid, 64 * kChainWaves, (hipStream_t)stream, a);
  return check_launch("gated_delta_bwd16_chain");
}

extern "C" int atma_gated_delta_bwd16_local(const void* q, const void* k, const void* v, const void* d_out,
                                            const float* f, const void* s_entry, const void* ds_end, const void* u,
                                            const float* dy, void* dq, void* dk, void* dv, float* dg, float* dbeta,
                                            int64_t B, int64_t T, int64_t H, int64_t Hkv, int64_t d, int dtype,
                                            void* stream) {
  using namespace atma;
  if (!bwd16_dims_ok(d, dtype, "gated_delta_bwd16_local")) return ATMA_ERR_UNSUPPORTED;
  if (B < 0 || T < 0 || H <= 0 || Hkv <= 0 || H % Hkv) return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_local: bad sizes");
  const int64_t NC = (T + 63) / 64;
  if (B == 0 || NC == 0) return ATMA_OK;
  if (!q || !k || !v || !d_out || !f || !s_entry || !ds_end || !u || !dy || !dq || !dk || !dv || !dg || !dbeta)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_local: null pointer");
  if (!aligned16({q, k, v, d_out, s_entry, ds_end, u, dy, dq, dk, dv}))
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_local: operands must be 16-byte aligned");
  if (B * H * NC > 0x7fffffff || B * T > 0x7fffffff)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_local: sizes too large");
  Bwd16LocalArgs a{q, d_out, k, v, f, s_entry, ds_end, u, dy, dq, dk, dv, dg, dbeta,
                   (int)B, (int)T, (int)H, (int)NC, (int)(H / Hkv)};
  const dim3 grid((unsigned)(B * H * NC));
  ATMA_BWD16_DISPATCH(gdn_bwd16_local_kernel, grid, (hipStream_t)stream, a);
  return check_launch("gated_delta_bwd16_local");
}

extern "C" int atma_gated_delta_bwd16_group_sum(const void* dk, const void* dv, void* dk_out, void* dv_out,
                                                int64_t rows, int64_t H, int64_t Hkv, int64_t d, int dtype,
                                                void* stream) {
  using namespace atma;
  if (!bwd16_dims_ok(d, dtype, "gated_delta_bwd16_group_sum")) return ATMA_ERR_UNSUPPORTED;
  if (rows < 0 || Hkv <= 0 || H <= 0 || H % Hkv)
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_group_sum: bad sizes");
  if (rows == 0) return ATMA_OK;
  if (!dk || !dv || !dk_out || !dv_out || !aligned16({dk, dv, dk_out, dv_out}))
    return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_group_sum: null or misaligned pointer");
  const int64_t n = rows * Hkv * d / 8;
  if (n > 0x7fffffffll * 256) return set_error(ATMA_ERR_INVALID, "gated_delta_bwd16_group_sum: sizes too large");
  const dim3 grid((unsigned)((n + 255) / 256), 2);
  hipStream_t s = (hipStream_t)stream;
  const auto *pk = (const u32x4*)dk, *pv = (const u32x4*)dv;
  auto *ok = (u32x4*)dk_out, *ov = (u32x4*)dv_out;
  const int G = (int)(H / Hkv), cpr = (int)(d / 8);
  if (dtype == ATMA_BF16) gdn_bwd16_group_sum_kernel<bf16><<<grid, dim3(256), 0, s>>>(pk, pv, ok, ov, n, G, cpr);
  else gdn_bwd16_group_sum_kernel<f16><<<grid, dim3(256), 0, s>>>(pk, pv, ok, ov, n, G, cpr);
  return check_launch("gated_delta_bwd16_group_sum");
}
