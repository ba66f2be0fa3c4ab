// Chunked gated-delta prefill with state carry (FLA chunk_gated_delta_rule contract).
//
// Reference arithmetic: gated_delta_chunked, model/blocks.py:375-423 (UT form,
// chunk C; decay first, undecayed write, self-inclusive readout), called through
// the FLA signature at model/blocks.py:44-49 and inference/models/atma.py:285-287.
//
// With lg_p = sum_{l<=p} g_l (g = log gamma) inside a chunk, ge_p = exp(lg_p),
// A[p,s] = beta_p exp(lg_p - lg_s) k_p.k_s (s < p) and T = (I + A)^-1 (unit lower
// triangular), the UT solve of the reference is folded into state-independent
// per-chunk operands (the WY form):
//     W  = T diag(beta ge) K          U0 = T diag(beta) V
//     Rq[p,s] = exp(lg_p - lg_s) q_p.k_s (s <= p)
//     Qt = diag(ge) Q - Rq W          R0 = Rq U0
//     Kd = diag(exp(lg_C - lg_s)) K   gC = exp(lg_C)
// after which one chunk of the recurrence on the [K, V] state S is
//     U = U0 - W S,   O = Qt S + R0,   S <- gC S + Kd^T U.
//
// Pass 1 (prep) is parallel over every (sequence, head, chunk); pass 2 runs the
// chunks in order, parallel over (sequence, head) x 16-column slabs of S (the
// state columns are independent), with the slab in registers for the whole
// sequence.  All arithmetic is fp32, the products on v_mfma_f32_16x16x4f32 (which
// rounds as fp32 fused multiply-adds do) with the contraction index permuted, step 4 j + e
// taking k = 16 j + 4 g + e, so that a lane's A operand comes as 16-byte reads of its row.
#include <algorithm>

#include "gated_delta.h"

namespace atma {

template <int D>
__host__ __device__ constexpr int64_t gdn_rec_floats() {
  return 5 * (int64_t)kChunk * D + 4;
}

// One workgroup of four waves per (sequence, head, chunk).  Wave P forms row block P of K K^T and Q K^T, wave 0 inverts
// I + A by 16 x 16 blocks, then wave w takes d columns [D/4 w, D/4 (w + 1)) of the records: W and U0, whose accumulators
// are the next product's B operand as they stand.  Bound by latency, one workgroup per CU (its rows in LDS): 2,048
// tokens of 8 heads, d = 128 42 us; 104 with the products on VALU and the inverse column by column.
template <typename T, int D>
__global__ void __launch_bounds__(256, 1) gdn_prep_kernel(GdnArgs a) {
  constexpr int C = kChunk, P = D + 4, PC = C + 4;
  constexpr int KJ = D / 16, DL = D / 64;  // 16-wide k blocks over D; elements of a row per lane
  __shared__ __attribute__((aligned(16))) float Ks[C * P], Qs[C * P], Vs[C * P];
  __shared__ __attribute__((aligned(16))) float Tl[C * PC], Rl[C * PC];  // N = A, then T; Rq
  __shared__ __attribute__((aligned(16))) float Nd[4 * 256];            // diagonal blocks of N^T, then of T^T
  __shared__ __attribute__((aligned(16))) float lg[C], bet[C], bge[C], tail[C], ge[C];

  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = blockIdx.x, bh = blockIdx.y;
  const int b = bh / a.H, h = bh % a.H;
  const int t0 = c * C;

  // ---- rows, all loads first: L2-normalise q/k, scale q; padded rows are zero with g = beta = 0
  {
    float qv[16][DL], kv[16][DL], vv[16][DL];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = t0 + wave + 4 * i;
      const bool ok = t < a.T;
      const T* qr = (const T*)a.q + b * a.q_sb + (int64_t)t * a.q_st + h * a.q_sh;
      const T* kr = (const T*)a.k + b * a.k_sb + (int64_t)t * a.k_st + (h / a.G) * a.k_sh;
      const T* vr = (const T*)a.v + b * a.v_sb + (int64_t)t * a.v_st + (h / a.G) * a.v_sh;
#pragma unroll
      for (int e = 0; e < DL; ++e) {
        qv[i][e] = ok ? to_f32(qr[lane + 64 * e]) : 0.f;
        kv[i][e] = ok ? to_f32(kr[lane + 64 * e]) : 0.f;
        vv[i][e] = ok ? to_f32(vr[lane + 64 * e]) : 0.f;
      }
    }
    float gl = 0.f, bt = 0.f;
    if (wave == 0 && t0 + lane < a.T) {
      const int64_t gi = ((int64_t)b * a.T + t0 + lane) * a.H + h;
      gl = gdn_load_g(a, gi);
      bt = gdn_load_beta(a, gi);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = wave + 4 * i;
      float iq = 1.f, ik = 1.f;
      if (a.l2norm) {
        float qq = 0.f, kk = 0.f;
#pragma unroll
        for (int e = 0; e < DL; ++e) {
          qq += qv[i][e] * qv[i][e];
          kk += kv[i][e] * kv[i][e];
        }
        iq = 1.f / fmaxf(sqrtf(wave_sum(qq)), 1e-12f);
        ik = 1.f / fmaxf(sqrtf(wave_sum(kk)), 1e-12f);
      }
#pragma unroll
      for (int e = 0; e < DL; ++e) {
        Qs[r * P + lane + 64 * e] = qv[i][e] * iq * a.scale;
        Ks[r * P + lane + 64 * e] = kv[i][e] * ik;
        Vs[r * P + lane + 64 * e] = vv[i][e];
      }
    }
    if (wave == 0) {  // inclusive log decays and the per-token factors
      float x = gl;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
      }
      const float e = expf(x);
      lg[lane] = x;
      bet[lane] = bt;
      ge[lane] = e;
      bge[lane] = bt * e;
      tail[lane] = expf(__shfl(x, 63, 64) - x);
    }
  }
  __syncthreads();

  auto row4 = [&](const float* tile, int pitch, int row0, int k0) {  // A operand (or B of the transpose): 4 k of a row
    return *(const f32x4*)(tile + (row0 + c16) * pitch + k0 + 4 * g);
  };
  auto mac4 = [&](const f32x4& x, const f32x4& y, f32x4 acc) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], acc, 0, 0, 0);
    return acc;
  };
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};

  // ---- row block R = wave of N = A (strictly lower, scaled by beta_p) and Rq (lower): row p = 16 R + 4 g + i, column
  // s = 16 S + c16
  {
    const int R = wave;
    f32x4 ka[KJ], qa[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      ka[j] = row4(Ks, P, 16 * R, 16 * j);
      qa[j] = row4(Qs, P, 16 * R, 16 * j);
    }
#pragma unroll
    for (int S = 0; S < 4; ++S) {
      if (S > R) break;
      f32x4 kk[2] = {z, z}, qk[2] = {z, z};
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        const f32x4 kb = row4(Ks, P, 16 * S, 16 * j);
        kk[j & 1] = mac4(ka[j], kb, kk[j & 1]);
        qk[j & 1] = mac4(qa[j], kb, qk[j & 1]);
      }
      const int sc = 16 * S + c16;
      f32x4 n;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = 16 * R + 4 * g + i;
        const float dec = sc <= p ? expf(lg[p] - lg[sc]) : 0.f;
        n[i] = sc < p ? bet[p] * dec * (kk[0][i] + kk[1][i]) : 0.f;
        Tl[p * PC + sc] = n[i];
        Rl[p * PC + sc] = sc <= p ? dec * (qk[0][i] + qk[1][i]) : 0.f;
      }
      if (S == R) *(f32x4*)(Nd + R * 256 + c16 * 16 + 4 * g) = n;  // N^T rows
    }
  }
  __syncthreads();

  // ---- T = (I + N)^-1 (wave 0): the diagonal blocks by forward substitution, lane (g, c) solving column c of block g;
  // below them, level L = P - S, T_PS = -T_PP sum_{k=S}^{P-1} N_Pk T_kS by block products (left factors transposed)
  if (wave == 0) {
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
      wave_sync();
      float* mt = Nd + g * 256 + c16 * 16;  // T^T row c = column c of T
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) *(f32x4*)(mt + 4 * q4) = f32x4{x[4 * q4], x[4 * q4 + 1], x[4 * q4 + 2], x[4 * q4 + 3]};
    }
    wave_sync();
    f32x4 tpp[4], tppT[4];  // T_PP and T_PP^T in the accumulator layout
#pragma unroll
    for (int B = 0; B < 4; ++B) {
      tpp[B] = *(const f32x4*)(Nd + B * 256 + c16 * 16 + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) tppT[B][i] = Nd[B * 256 + (4 * g + i) * 16 + c16];
    }
    auto nt = [&](int S, int B) { return row4(Tl, PC, 16 * B, 16 * S); };  // block (B, S) of N, transposed layout
    const f32x4 n10 = nt(0, 1), n20 = nt(0, 2), n30 = nt(0, 3), n21 = nt(1, 2), n31 = nt(1, 3), n32 = nt(2, 3);
    const f32x4 y10 = blk_mul(n10, tpp[0], z), y21 = blk_mul(n21, tpp[1], z), y32 = blk_mul(n32, tpp[2], z);
    const f32x4 t10 = -blk_mul(tppT[1], y10, z), t21 = -blk_mul(tppT[2], y21, z);
    const f32x4 tt01 = -blk_mul(y10, tppT[1], z), tt12 = -blk_mul(y21, tppT[2], z), tt23 = -blk_mul(y32, tppT[3], z);
    const f32x4 y20 = blk_mul(n21, t10, blk_mul(n20, tpp[0], z)), y31 = blk_mul(n32, t21, blk_mul(n31, tpp[1], z));
    const f32x4 t20 = -blk_mul(tppT[2], y20, z);
    const f32x4 tt02 = -blk_mul(y20, tppT[2], z), tt13 = -blk_mul(y31, tppT[3], z);
    const f32x4 y30 = blk_mul(n32, t20, blk_mul(n31, t10, blk_mul(n30, tpp[0], z)));
    const f32x4 tt03 = -blk_mul(y30, tppT[3], z);
    wave_sync();
    // the transposed-form block (S, B) is row 16 B + c, columns 16 S + 4 g .. + 3 of T; the blocks above stay unread
    const f32x4 tb[4][4] = {{tppT[0], z, z, z}, {tt01, tppT[1], z, z}, {tt02, tt12, tppT[2], z}, {tt03, tt13, tt23, tppT[3]}};
#pragma unroll
    for (int B = 0; B < 4; ++B)
#pragma unroll
      for (int S = 0; S <= B; ++S) *(f32x4*)(Tl + (16 * B + c16) * PC + 16 * S + 4 * g) = tb[B][S];
  }
  __syncthreads();

  // ---- the records' d columns 16 n + c16 of wave w
  float* rec = (float*)a.ws + ((int64_t)bh * a.NC + c) * gdn_rec_floats<D>();
  if (tid == 0) rec[5 * C * D] = ge[C - 1];
#pragma unroll
  for (int nn = 0; nn < DL; ++nn) {
    const int d = 16 * (DL * wave + nn) + c16;
    f32x4 kb[4], vb[4];  // B operands, k = s = 16 j + 4 g + e: diag(beta ge) K and diag(beta) V
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 bk = *(const f32x4*)(bge + 16 * j + 4 * g), bv = *(const f32x4*)(bet + 16 * j + 4 * g);
      const f32x4 tl = *(const f32x4*)(tail + 16 * j + 4 * g);
      f32x4 kd;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int s = 16 * j + 4 * g + e;
        const float kx = Ks[s * P + d];
        kb[j][e] = kx * bk[e];
        vb[j][e] = Vs[s * P + d] * bv[e];
        kd[e] = tl[e] * kx;
      }
      *(f32x4*)(rec + 4 * C * D + d * C + 16 * j + 4 * g) = kd;
    }
    f32x4 w[4], u[4];
#pragma unroll
    for (int B = 0; B < 4; ++B) {
      w[B] = u[B] = z;
#pragma unroll
      for (int j = 0; j <= B; ++j) {
        const f32x4 t = row4(Tl, PC, 16 * B, 16 * j);
        w[B] = mac4(t, kb[j], w[B]);
        u[B] = mac4(t, vb[j], u[B]);
      }
    }
#pragma unroll
    for (int B = 0; B < 4; ++B) {
      f32x4 qt = z, r0 = z;
#pragma unroll
      for (int j = 0; j <= B; ++j) {
        const f32x4 r = row4(Rl, PC, 16 * B, 16 * j);
        qt = mac4(r, w[j], qt);
        r0 = mac4(r, u[j], r0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = 16 * B + 4 * g + i;
        rec[p * D + d] = w[B][i];
        rec[C * D + p * D + d] = u[B][i];
        rec[2 * C * D + p * D + d] = ge[p] * Qs[p * P + d] - qt[i];
        rec[3 * C * D + p * D + d] = r0[i];
      }
    }
  }
}

// One workgroup of four waves per (sequence-head, 16 state columns): wave w owns 16 tokens of U and O and D / 4 rows of
// the state.  The state and U pass between the waves through LDS (two barriers a chunk); the records come straight into
// operand registers, each part loaded for the next chunk as soon as this one's is consumed; O's product, off the chain,
// runs while U is exchanged.  Bound by the chain of a chunk, D / 4 products and 2 exchanges: 2,048 tokens of 8 heads,
// d = 128 111 us; 355 with the records staged through LDS and the products on VALU.
template <typename T, int D>
__global__ void __launch_bounds__(256, 1) gdn_scan_kernel(GdnArgs a) {
  constexpr int C = kChunk, VS = 16, KJ = D / 16, RT = D / 64;
  __shared__ __attribute__((aligned(16))) float Sl[VS * (D + 4)], Ul[VS * (C + 4)];  // [column][row]
  gdn_signal_start(a);

  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.x, v0 = blockIdx.y * VS;
  const int b = bh / a.H, h = bh % a.H;
  const int p0 = 16 * wave + 4 * g;  // the lane's tokens p0 + i

  f32x4 S[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      S[t][i] = a.s0 ? a.s0[((int64_t)bh * D + 16 * (RT * wave + t) + 4 * g + i) * D + v0 + c16] : 0.f;

  f32x4 w[KJ], q[KJ], kd[RT][4], u0, r0;
  float gC;
  const float* rec0 = (const float*)a.ws + (int64_t)bh * a.NC * gdn_rec_floats<D>();
  auto load_w = [&](const float* rec) {
#pragma unroll
    for (int j = 0; j < KJ; ++j) w[j] = *(const f32x4*)(rec + (16 * wave + c16) * D + 16 * j + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) u0[i] = rec[C * D + (p0 + i) * D + v0 + c16];
  };
  auto load_q = [&](const float* rec) {
#pragma unroll
    for (int j = 0; j < KJ; ++j) q[j] = *(const f32x4*)(rec + 2 * C * D + (16 * wave + c16) * D + 16 * j + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) r0[i] = rec[3 * C * D + (p0 + i) * D + v0 + c16];
  };
  auto load_k = [&](const float* rec) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        kd[t][j] = *(const f32x4*)(rec + 4 * C * D + (16 * (RT * wave + t) + c16) * C + 16 * j + 4 * g);
    gC = rec[5 * C * D];
  };
  load_w(rec0);
  load_q(rec0);
  load_k(rec0);
  for (int c = 0; c < a.NC; ++c) {
    const float* next = rec0 + (int64_t)(c + 1) * gdn_rec_floats<D>();
    const bool more = c + 1 < a.NC;
#pragma unroll
    for (int t = 0; t < RT; ++t) *(f32x4*)(Sl + c16 * (D + 4) + 16 * (RT * wave + t) + 4 * g) = S[t];
    __syncthreads();  // the state is whole; every wave is done with the previous U
    f32x4 sv[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j) sv[j] = *(const f32x4*)(Sl + c16 * (D + 4) + 16 * j + 4 * g);
    f32x4 x[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}}, o[2] = {r0, x[0]};
#pragma unroll
    for (int j = 0; j < KJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][e], sv[j][e], x[e & 1], 0, 0, 0);
    *(f32x4*)(Ul + c16 * (C + 4) + p0) = u0 - (x[0] + x[1]);
    if (more) load_w(next);
#pragma unroll
    for (int j = 0; j < KJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[j][e], sv[j][e], o[e & 1], 0, 0, 0);
    if (more) load_q(next);
    __syncthreads();  // U is whole; every wave has read the state
    f32x4 uv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) uv[j] = *(const f32x4*)(Ul + c16 * (C + 4) + 16 * j + 4 * g);
#pragma unroll
    for (int t = 0; t < RT; ++t) S[t] *= gC;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < RT; ++t) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kd[t][j][e], uv[j][e], S[t], 0, 0, 0);
    if (more) load_k(next);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = c * C + p0 + i;
      if (t < a.T) ((T*)a.o)[(((int64_t)b * a.T + t) * a.H + h) * D + v0 + c16] = from_f32<T>(o[0][i] + o[1][i]);
    }
  }
  if (a.s_out) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a.s_out[((int64_t)bh * D + 16 * (RT * wave + t) + 4 * g + i) * D + v0 + c16] = S[t][i];
  }
}

template <typename T, int D>
static int launch_gdn(GdnArgs a, hipStream_t s) {
  gdn_prep_kernel<T, D><<<dim3((unsigned)a.NC, (unsigned)(a.B * a.H)), dim3(256), 0, s>>>(a);
  int rc = check_launch("chunk_gated_delta_rule(prep)");
  if (rc) return rc;
  gdn_scan_kernel<T, D><<<dim3((unsigned)(a.B * a.H), D / 16), dim3(256), 0, s>>>(a);
  return check_launch("chunk_gated_delta_rule(scan)");
}

}  // namespace atma

extern "C" size_t atma_chunk_gated_delta_workspace_bytes(int64_t B, int64_t T, int64_t H,
                                                         int64_t dk, int64_t dv, int64_t chunk,
                                                         int dtype) {
  (void)dv;
  if (B <= 0 || T <= 0 || H <= 0 || chunk != atma::kChunk || (dk != 64 && dk != 128)) return 0;
  const int64_t nc = (T + chunk - 1) / chunk;
  if (dtype == ATMA_BF16 || dtype == ATMA_F16)
    return atma::gdn16_workspace_bytes(B * H, nc, (int)dk);
  const int64_t rec = 5 * chunk * dk + 4;
  return (size_t)(B * H * nc * rec) * sizeof(float);
}

extern "C" int atma_chunk_gated_delta_rule(
    const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sb,
    int64_t k_st, int64_t k_sh, const void* v, int64_t v_sb, int64_t v_st, int64_t v_sh,
    const float* g, const float* beta, const float* initial_state, float* final_state, void* o,
    int64_t B, int64_t T, int64_t H, int64_t Hkv, int64_t dk, int64_t dv, int dtype, float scale,
    int use_qk_l2norm, int gate_logits, float g_bias, float b_bias, int64_t chunk, void* workspace,
    size_t workspace_bytes, int32_t* start_flag, int32_t start_epoch, void* stream) {
  using namespace atma;
  if (chunk != kChunk)
    return set_error(ATMA_ERR_UNSUPPORTED, "chunk_gated_delta_rule: chunk must be %d", kChunk);
  if (dk != dv || (dk != 64 && dk != 128))
    return set_error(ATMA_ERR_UNSUPPORTED, "chunk_gated_delta_rule: dk=dv in {64,128} (got %lld,%lld)",
                     (long long)dk, (long long)dv);
  if (B < 0 || T < 0 || H <= 0) return set_error(ATMA_ERR_INVALID, "chunk_gated_delta_rule: bad sizes");
  if (Hkv <= 0 || H % Hkv)
    return set_error(ATMA_ERR_INVALID, "chunk_gated_delta_rule: H=%lld not a multiple of Hkv=%lld",
                     (long long)H, (long long)Hkv);
  if (B * H > 0x7fffffffll || T > (1ll << 30))
    return set_error(ATMA_ERR_INVALID, "chunk_gated_delta_rule: sizes too large");
  const int es = dtype_size(dtype);
  if (!es) return set_error(ATMA_ERR_INVALID, "chunk_gated_delta_rule: unknown dtype %d", dtype);
  if (B == 0) return ATMA_OK;
  if (T == 0) {
    // no tokens: the final state is the initial state -- not representable without a copy
    // kernel; callers short-circuit T == 0 on the host.
    return set_error(ATMA_ERR_INVALID, "chunk_gated_delta_rule: T must be > 0");
  }
  if (!q || !k || !v || !g || !beta || !o)
    return set_error(ATMA_ERR_INVALID, "chunk_gated_delta_rule: null pointer");
  if (es == 2 && T * H * dk * 2 >= (1ll << 32))  // one sequence's output rows form one buffer
    return set_error(ATMA_ERR_UNSUPPORTED, "chunk_gated_delta_rule: T*H*d too large for one sequence");
  if (es == 2 && (q_st >= (1 << 24) || k_st >= (1 << 24) || v_st >= (1 << 24) || q_st < dk || k_st < dk ||
                  v_st < dv))
    // the kernels copy a chunk's q / k / v rows through one buffer descriptor each
    return set_error(ATMA_ERR_UNSUPPORTED, "chunk_gated_delta_rule: q/k/v token stride out of range");
  if (es == 2 && B * H * ((T + 63) / 64) >= (1ll << 31))  // the prep kernel indexes items in 32 bits
    return set_error(ATMA_ERR_UNSUPPORTED, "chunk_gated_delta_rule: B*H*chunks too large");
  const size_t need = atma_chunk_gated_delta_workspace_bytes(B, T, H, dk, dv, chunk, dtype);
  if (!workspace || workspace_bytes < need)
    return set_error(ATMA_ERR_WORKSPACE, "chunk_gated_delta_rule: workspace %zu < %zu bytes",
                     workspace_bytes, need);
  GdnArgs a{};
  a.q = q; a.q_sb = q_sb; a.q_st = q_st; a.q_sh = q_sh;
  a.k = k; a.k_sb = k_sb; a.k_st = k_st; a.k_sh = k_sh;
  a.v = v; a.v_sb = v_sb; a.v_st = v_st; a.v_sh = v_sh;
  a.g = g; a.beta = beta; a.s0 = initial_state; a.s_out = final_state; a.o = o;
  a.B = (int)B; a.T = (int)T; a.H = (int)H; a.NC = (int)((T + chunk - 1) / chunk);
  a.G = (int)(H / Hkv);
  a.scale = scale; a.l2norm = use_qk_l2norm ? 1 : 0; a.ws = workspace;
  a.gate_logits = gate_logits ? 1 : 0; a.g_bias = g_bias; a.b_bias = b_bias;
  a.start_flag = start_flag; a.start_epoch = start_epoch;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == ATMA_BF16 || dtype == ATMA_F16) return launch_gdn16(a, nullptr, dtype, (int)dk, s);
  return dk == 128 ? launch_gdn<float, 128>(a, s) : launch_gdn<float, 64>(a, s);
}

namespace atma {
// A ragged launch scans every sequence plainly, so its longest one sets the time.  Sequences long enough to split (64
// chunks; one of 4,096 tokens and 8 heads then takes about half the time, two of them in turn already as long as one
// plain launch of both) are split one after another where that takes less: all their halves against the longest.
static bool gdn_long(int64_t H, int64_t d, int64_t T) {
  const int64_t chunks = (T + kChunk - 1) / kChunk;
  int64_t states;
  return chunks >= 64 && gdn16_segments(H, chunks, (int)d, 256, states) >= 4;
}
static bool gdn_split_long(int64_t B, int64_t H, int64_t d, const int64_t* seq_lens) {
  int64_t longest = 0, sum = 0;
  for (int64_t b = 0; b < B; ++b)
    if (gdn_long(H, d, seq_lens[b])) {
      longest = std::max(longest, seq_lens[b]);
      sum += seq_lens[b];
    }
  return sum > 0 && sum < 2 * longest;
}
}  // namespace atma

extern "C" size_t atma_gated_delta_prefill_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t d,
                                                           const int64_t* seq_lens) {
  using namespace atma;
  if (B <= 0 || H <= 0 || (d != 64 && d != 128)) return 0;
  if (!seq_lens) return T > 0 ? gdn16_workspace_bytes(B * H, (T + kChunk - 1) / kChunk, (int)d) : 0;
  int64_t most = 0;  // the launches of kVarSeqs sequences follow each other in the same workspace
  for (int64_t b0 = 0; b0 < B; b0 += kVarSeqs) {
    int64_t chunks = 0;
    for (int64_t b = b0; b < B && b < b0 + kVarSeqs; ++b) chunks += seq_lens[b] > 0 ? (seq_lens[b] + kChunk - 1) / kChunk : 0;
    most = std::max(most, chunks);
  }
  size_t bytes = (size_t)(most * H) * (size_t)kGdn16RecBytes;
  if (gdn_split_long(B, H, d, seq_lens))
    for (int64_t b = 0; b < B; ++b)
      if (gdn_long(H, d, seq_lens[b]))
        bytes = std::max(bytes, gdn16_workspace_bytes(H, (seq_lens[b] + kChunk - 1) / kChunk, (int)d));
  return bytes;
}

extern "C" int atma_gated_delta_prefill(
    const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sb, int64_t k_st, int64_t k_sh,
    const void* v, int64_t v_sb, int64_t v_st, int64_t v_sh, const float* g, const float* beta, float* state_table,
    const int64_t* slots, int64_t num_slots, void* o, int64_t B, int64_t T, const int64_t* seq_lens, int64_t H,
    int64_t Hkv, int64_t d, int dtype, float scale, int use_qk_l2norm, int gate_logits, float g_bias, float b_bias,
    void* workspace, size_t workspace_bytes, int32_t* start_flag, int32_t start_epoch, void* stream) {
  using namespace atma;
  if (dtype != ATMA_BF16 && dtype != ATMA_F16)
    return set_error(ATMA_ERR_UNSUPPORTED, "gated_delta_prefill: 16-bit rows only (dtype %d)", dtype);
  if (d != 64 && d != 128) return set_error(ATMA_ERR_UNSUPPORTED, "gated_delta_prefill: d 64 or 128");
  if (B < 0 || H <= 0 || Hkv <= 0 || H % Hkv || num_slots < 0 || num_slots > 0x7fffffff || (!seq_lens && T < 1) ||
      B * H > 0x7fffffff)
    return set_error(ATMA_ERR_INVALID, "gated_delta_prefill: bad sizes");
  if (B == 0) return ATMA_OK;
  if (!q || !k || !v || !g || !beta || !state_table || !slots || !o)
    return set_error(ATMA_ERR_INVALID, "gated_delta_prefill: null pointer");
  if (q_st >= (1 << 24) || k_st >= (1 << 24) || v_st >= (1 << 24) || q_st < d || k_st < d || v_st < d)
    return set_error(ATMA_ERR_UNSUPPORTED, "gated_delta_prefill: q/k/v token stride out of range");
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) % 16 ||
      (q_sb | q_st | q_sh | k_sb | k_st | k_sh | v_sb | v_st | v_sh) % 8)
    return set_error(ATMA_ERR_INVALID, "gated_delta_prefill: rows must be 16-byte aligned");
  int64_t longest = T, total = 0;
  if (seq_lens) {
    longest = 0;
    for (int64_t b = 0; b < B; ++b) {
      if (seq_lens[b] < 0) return set_error(ATMA_ERR_INVALID, "gated_delta_prefill: negative sequence length");
      longest = std::max(longest, seq_lens[b]);
      total += seq_lens[b];
    }
    if (total == 0) return ATMA_OK;
  }
  const int64_t chunks = (longest + kChunk - 1) / kChunk;
  if (longest > 1 << 30 || total > 1 << 30 || longest * H * d * 2 >= (1ll << 32) ||
      std::min<int64_t>(B, seq_lens ? kVarSeqs : B) * H * chunks >= (1ll << 31))
    return set_error(ATMA_ERR_UNSUPPORTED, "gated_delta_prefill: sizes too large");
  if (!workspace || workspace_bytes < atma_gated_delta_prefill_workspace_bytes(B, T, H, d, seq_lens))
    return set_error(ATMA_ERR_WORKSPACE, "gated_delta_prefill: workspace too small");
  GdnArgs a{};
  a.q = q; a.q_sb = q_sb; a.q_st = q_st; a.q_sh = q_sh;
  a.k = k; a.k_sb = k_sb; a.k_st = k_st; a.k_sh = k_sh;
  a.v = v; a.v_sb = v_sb; a.v_st = v_st; a.v_sh = v_sh;
  a.g = g; a.beta = beta; a.s0 = state_table; a.s_out = state_table; a.o = o;
  a.B = (int)B; a.T = (int)T; a.H = (int)H; a.NC = (int)chunks;
  a.G = (int)(H / Hkv);
  a.scale = scale; a.l2norm = use_qk_l2norm ? 1 : 0; a.ws = workspace;
  a.gate_logits = gate_logits ? 1 : 0; a.g_bias = g_bias; a.b_bias = b_bias;
  a.start_flag = start_flag; a.start_epoch = start_epoch;
  a.slots = slots; a.num_slots = num_slots;
  hipStream_t s = (hipStream_t)stream;
  if (!seq_lens) return launch_gdn16(a, nullptr, dtype, (int)d, s);
  const bool split = gdn_split_long(B, H, d, seq_lens);
  int64_t start = 0;
  for (int64_t b0 = 0; b0 < B; b0 += kVarSeqs) {
    int order[kVarSeqs], starts[kVarSeqs], n = 0;
    for (int64_t b = b0; b < B && b < b0 + kVarSeqs; ++b) {
      starts[b - b0] = (int)start;
      if (split && gdn_long(H, d, seq_lens[b])) {
        GdnArgs l = a;
        l.q = (const char*)q + start * q_st * 2;
        l.k = (const char*)k + start * k_st * 2;
        l.v = (const char*)v + start * v_st * 2;
        l.g = g + start * H;
        l.beta = beta + start * H;
        l.o = (char*)o + start * H * d * 2;
        l.slots = slots + b;
        l.B = 1; l.T = (int)seq_lens[b]; l.NC = (int)((seq_lens[b] + kChunk - 1) / kChunk);
        const int rc = launch_gdn16(l, nullptr, dtype, (int)d, s);
        if (rc) return rc;
      } else if (seq_lens[b] > 0) {
        order[n++] = (int)(b - b0);
      }
      start += seq_lens[b];
    }
    if (n == 0) continue;
    std::stable_sort(order, order + n, [&](int x, int y) { return seq_lens[b0 + x] > seq_lens[b0 + y]; });
    VarSeqs vs{};
    vs.n = n;
    for (int i = 0, c = 0; i < n; ++i) {
      vs.start[i] = starts[order[i]];
      vs.len[i] = (int)seq_lens[b0 + order[i]];
      vs.chunk0[i] = c;
      vs.row[i] = (int)b0 + order[i];
      c += (vs.len[i] + kChunk - 1) / kChunk;
    }
    const int rc = launch_gdn16(a, &vs, dtype, (int)d, s);
    if (rc) return rc;
  }
  return ATMA_OK;
}

namespace atma {

// One lane polls the flag (agent-scope loads, which see another kernel's store across the
// XCDs' L2s) with a sleep between polls, and gives up after limit_ticks of the constant
// wall clock, so the kernel always ends; a timeout only costs the overlap, never results.
__global__ void __launch_bounds__(64) start_wait_kernel(const int* flag, int epoch, uint64_t limit_ticks) {
  if (threadIdx.x != 0) return;
  const uint64_t t0 = wall_clock64();
  while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch) {
    if (wall_clock64() - t0 > limit_ticks) break;
    __builtin_amdgcn_s_sleep(2);
  }
}

}  // namespace atma

extern "C" int atma_wait_start_flag(const int32_t* flag, int32_t epoch, int64_t timeout_us, void* stream) {
  using namespace atma;
  if (!flag) return set_error(ATMA_ERR_INVALID, "wait_start_flag: null flag");
  if (timeout_us <= 0 || timeout_us > 10000000)
    return set_error(ATMA_ERR_INVALID, "wait_start_flag: timeout_us must be in (0, 1e7]");
  static int rate_khz = 0;  // wall clock rate; the same for every MI355X device
  if (!rate_khz) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || rate_khz <= 0)
      return set_error(ATMA_ERR_HIP, "wait_start_flag: wall clock rate unavailable");
  }
  const uint64_t ticks = (uint64_t)timeout_us * (uint64_t)rate_khz / 1000u;
  start_wait_kernel<<<dim3(1), dim3(64), 0, (hipStream_t)stream>>>(flag, epoch, ticks);
  return check_launch("wait_start_flag");
}
