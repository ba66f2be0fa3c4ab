// Chunked gated-delta prefill for bf16 / fp16 inputs on MFMA (v_mfma_f32_16x16x32).
//
// Algebra of gated_delta_chunked (model/blocks.py:375-423; FLA convention: decay
// first, undecayed write, self-inclusive readout).  Inside a 64-token chunk with
// inclusive log-decays lg_p, ge_p = exp(lg_p), row weights ik = 1 / |k|, iq = scale / |q|,
// A[p,s] = beta_p exp(lg_p - lg_s) kn_p.kn_s (s < p) and T = (I + A)^-1, the carried state
// S ([K, V]) gives
//     U = T diag(beta) (V - diag(ge ik) K S)                      (raw k rows K)
//     O = diag(ge iq) Q S + Rq U,          Rq[p,s] = exp(lg_p - lg_s) qn_p.kn_s (s <= p)
//     S <- exp(lg_C) S + K^T diag(exp(lg_C - lg) ik) U
//
//  pass 1, gdn_prep16 -- one wave per (sequence, head, chunk) item, no workgroup
//    barriers: k and q rows straight from memory into MFMA fragments, row norms and the
//    log-decay prefix in registers, the Gram blocks K K^T and K Q^T on MFMA, T by forward
//    substitution on the 16 x 16 diagonal blocks (fp32, one lane per column) and three
//    levels of fp32 block products, then the record (T diag(beta) and Rq as MFMA
//    fragments, per-token factors; 14 KiB, layout in gated_delta.h).
//
//  pass 2, gdn_scan16_pair -- one workgroup of four waves per (sequence, head, 32-column
//    slab of the state).  The columns of the recurrence are independent: each of two chain
//    waves owns 16 whole columns and runs K S (16 MFMAs) -> X -> U = T diag(beta) X (6) ->
//    S update (16) in registers; each of two output waves computes the same columns'
//    O^T = S^T Q^T diag(geqs) + U^T Rq^T (22) from the state and U fragments the chain hands
//    over in LDS, and issues the copies: the k, q rows, the v slab and the record of chunk
//    c + 2 stream into a third LDS slot (direct buffer copies) while chunk c computes.  Two
//    workgroup barriers per chunk order the slots and the hand-over.  Segment summaries (no
//    output) run four such chain waves per workgroup, which issue the copies as well.
//
// Fragment layouts (v_mfma_f32_16x16x32: A lane (g, r) holds row r, k = 8g + [0, 8); B lane
// (g, c) holds column c, same k; accumulator lane (g, c) register i holds row 4g + i,
// column c).  State tile t of a wave holds rows k = 32 (t/2) + 8g + 4 (t%2) + i, so two
// tiles give the B fragment of k-step t/2 in natural k order.  Token contractions use the
// slot order 32 j + 4g + [0, 4), 32 j + 16 + 4g + [0, 4), which two accumulator tiles of
// consecutive 16-token blocks give without data movement; the record's fragments and the
// transposing LDS reads of k and v rows follow that order.
#include <algorithm>
#include <type_traits>

#include "gated_delta.h"

namespace atma {

__device__ __forceinline__ u32x4 lds16(const void* p) { return *(const u32x4*)p; }

// 16-bit element e (0..3) of an 8-byte vector, as float.
template <typename T>
__device__ __forceinline__ float elem16x2(const u32x2& x, int e) {
  const uint16_t u = (uint16_t)(x[e >> 1] >> ((e & 1) * 16));
  return (float)__builtin_bit_cast(T, u);
}

// acc + x.lo^2 + x.hi^2 for a packed pair of 16-bit values (v_dot2_f32_bf16 / _f16).
template <typename T>
__device__ __forceinline__ float dot2_sq(uint32_t x, float acc) {
  if constexpr (std::is_same_v<T, bf16>) {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    const v2 v = __builtin_bit_cast(v2, x);
    return __builtin_amdgcn_fdot2_f32_bf16(v, v, acc, false);
  } else {
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    const v2 v = __builtin_bit_cast(v2, x);
    return __builtin_amdgcn_fdot2(v, v, acc, false);
  }
}

// Eight floats (two accumulator tiles) -> one 16-byte MFMA fragment.
template <typename T>
__device__ __forceinline__ u32x4 pack8(const f32x4& lo, const f32x4& hi) {
  return u32x4{pack2<T>(lo[0], lo[1]), pack2<T>(lo[2], lo[3]), pack2<T>(hi[0], hi[1]), pack2<T>(hi[2], hi[3])};
}

// Sequence, head and chunk of a prep item (items: sequence by sequence, head by head, chunk by chunk); false past the last.
__device__ __forceinline__ bool gdn_item(const GdnArgs& a, const DenseSeqs&, uint32_t item, int& b, int& h, int& c) {
  if (item >= (uint32_t)(a.B * a.H * a.NC)) return false;
  const int bh = (int)(item / (uint32_t)a.NC);
  c = (int)(item % (uint32_t)a.NC);
  b = bh / a.H;
  h = bh % a.H;
  return true;
}
__device__ __forceinline__ bool gdn_item(const GdnArgs& a, const VarSeqs& v, uint32_t item, int& b, int& h, int& c) {
  const uint32_t chunk = item / (uint32_t)a.H;  // compare chunk counts: item < (chunk0 + NC) H
  int lo = 0, hi = v.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if ((uint32_t)v.chunk0[mid] <= chunk) lo = mid;
    else hi = mid - 1;
  }
  const uint32_t nc = (uint32_t)(v.len[lo] + 63) / 64, left = item - (uint32_t)v.chunk0[lo] * (uint32_t)a.H;
  b = lo;
  h = (int)(left / nc);
  c = (int)(left % nc);
  return h < a.H;
}

template <typename T, int D, typename SEQ>
__global__ void __launch_bounds__(256) gdn_prep16_kernel(GdnArgs a, SEQ seqs) {
  constexpr int C = kChunk, KS = D / 32;
  __shared__ __attribute__((aligned(16))) float Nb[4][4 * 256];  // per wave: N^T of the diagonal blocks
  __shared__ __attribute__((aligned(16))) float Mb[4][4 * 256];  // per wave: T^T of the diagonal blocks
  __shared__ __attribute__((aligned(16))) float Tk[4][6][C];     // per wave: per-token factors (below)

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const uint32_t item = blockIdx.x * 4u + (uint32_t)wave;  // B H NC < 2^31 (the entry checks)
  int b, h, c;
  if (!gdn_item(a, seqs, item, b, h, c)) return;             // a whole wave; the kernel has no barrier
  const SeqView sq = gdn_seq(a, seqs, b);
  const int rows = min(sq.T - c * C, C);
  float* tbt = Tk[wave][0];   // beta
  float* tik = Tk[wave][1];   // 1 / |k| (1 without l2norm, 0 past T)
  float* tiq = Tk[wave][2];   // scale / |q|
  // exponents (base 2) that fold the row-norm, write-strength and decay factors of a scaled
  // Gram entry into one exp2: aq = lg log2e + log2 iq, ak = lg log2e + log2(beta ik),
  // bk = lg log2e - log2 ik, so Rq[p,s] = exp2(aq_p - bk_s) q_p.k_s and A[p,s] =
  // exp2(ak_p - bk_s) k_p.k_s (a zero factor gives -inf / +inf, hence an exact 0)
  float* taq = Tk[wave][3];
  float* tak = Tk[wave][4];
  float* tbk = Tk[wave][5];
  float* nb = Nb[wave];
  float* mb = Mb[wave];
  char* rec = (char*)a.ws + (size_t)item * kGdn16RecBytes;

  // ---- k and q rows as MFMA fragments: lane (g, r) holds row 16p + r, columns 32s + 8g ..
  // (rows past T read as zeros)
  const auto krs = buffer_rsrc((const T*)a.k + sq.ko + (int64_t)c * C * a.k_st + (h / a.G) * a.k_sh,
                               (uint32_t)(((rows - 1) * a.k_st + D) * 2));
  const auto qrs = buffer_rsrc((const T*)a.q + sq.qo + (int64_t)c * C * a.q_st + h * a.q_sh,
                               (uint32_t)(((rows - 1) * a.q_st + D) * 2));
  u32x4 kf[4][KS], qf[4][KS];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      kf[p][s] = buffer_load16(krs, (uint32_t)(((16 * p + c16) * a.k_st + 32 * s + 8 * g) * 2), 0);
      qf[p][s] = buffer_load16(qrs, (uint32_t)(((16 * p + c16) * a.q_st + 32 * s + 8 * g) * 2), 0);
    }

  // ---- gates (lane = token) and the inclusive prefix sum of the log-decays
  float gl = 0.f, bt = 0.f;
  if (lane < rows) {
    const int64_t gi = (sq.tok0 + c * C + lane) * a.H + h;
    gl = gdn_load_g(a, gi);
    bt = gdn_load_beta(a, gi);
  }
  float lg = gl;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float y = __shfl_up(lg, off, 64);
    if (lane >= off) lg += y;
  }
  tbt[lane] = bt;

  // ---- row norms: partial sums over this lane's columns (packed pairs, v_dot2), then over
  // the four lane groups
  float nk[4], nq[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    nk[p] = nq[p] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        nk[p] = dot2_sq<T>(kf[p][s][e], nk[p]);
        nq[p] = dot2_sq<T>(qf[p][s][e], nq[p]);
      }
    nk[p] += __shfl_xor(nk[p], 16, 64);
    nq[p] += __shfl_xor(nq[p], 16, 64);
    nk[p] += __shfl_xor(nk[p], 32, 64);
    nq[p] += __shfl_xor(nq[p], 32, 64);
  }
  if (g == 0) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int row = 16 * p + c16;
      const bool ok = row < rows;
      tik[row] = ok ? (a.l2norm ? 1.f / fmaxf(sqrtf(nk[p]), 1e-12f) : 1.f) : 0.f;
      tiq[row] = ok ? (a.l2norm ? 1.f / fmaxf(sqrtf(nq[p]), 1e-12f) : 1.f) * a.scale : 0.f;
    }
  }
  wave_sync();

  // ---- per-token factors of the scan and the folded exponents
  {
    const float l2 = lg * kLog2e, ik = tik[lane], iq = tiq[lane];
    taq[lane] = l2 + __builtin_amdgcn_logf(iq);
    tak[lane] = l2 + __builtin_amdgcn_logf(bt * ik);
    tbk[lane] = l2 - __builtin_amdgcn_logf(ik);
    const float lgC = __shfl(lg, 63, 64);
    const float ge = __builtin_amdgcn_exp2f(lg * kLog2e);
    float* F = (float*)(rec + kGdn16F);
    F[lane] = __builtin_amdgcn_exp2f((lgC - lg) * kLog2e) * tik[lane];
    F[64 + lane] = ge * tik[lane];
    F[128 + lane] = ge * tiq[lane];
    if (lane == 0) F[192] = __builtin_amdgcn_exp2f(lgC * kLog2e);
  }

  // ---- Gram blocks on MFMA: gk(k, P) lane (g, c) register i = k_{16k+4g+i} . k_{16P+c},
  // gq(S, P) register i = k_{16S+4g+i} . q_{16P+c}
  f32x4 gk[10], gq[10];
#pragma unroll
  for (int P = 0; P < 4; ++P)
#pragma unroll
    for (int k = 0; k <= P; ++k) {
      f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        x = mfma16x16x32<T>(kf[k][s], kf[P][s], x);
        y = mfma16x16x32<T>(kf[k][s], qf[P][s], y);
      }
      gk[tri(k, P)] = x;
      gq[tri(k, P)] = y;
    }

  // ---- Rq, transposed: block (S, P) register i = Rq[16P + c][16S + 4g + i]; written as the
  // scan's B fragments (fragment (P, j) = blocks (2j, P), (2j + 1, P); blocks above the
  // diagonal are zero)
  {
    f32x4 rq[10];
#pragma unroll
    for (int P = 0; P < 4; ++P) {
      const int pt = 16 * P + c16;
      const float ap = taq[pt];
#pragma unroll
      for (int S = 0; S <= P; ++S) {
        const f32x4 bs = *(const f32x4*)(tbk + 16 * S + 4 * g);
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[i] = (16 * S + 4 * g + i <= pt) ? __builtin_amdgcn_exp2f(ap - bs[i]) * gq[tri(S, P)][i] : 0.f;
        rq[tri(S, P)] = v;
      }
    }
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    u32x4* Rb = (u32x4*)(rec + kGdn16Rb);
    Rb[0 * 64 + lane] = pack8<T>(rq[tri(0, 0)], z);
    Rb[1 * 64 + lane] = pack8<T>(rq[tri(0, 1)], rq[tri(1, 1)]);
    Rb[2 * 64 + lane] = pack8<T>(rq[tri(0, 2)], rq[tri(1, 2)]);
    Rb[3 * 64 + lane] = pack8<T>(rq[tri(2, 2)], z);
    Rb[4 * 64 + lane] = pack8<T>(rq[tri(0, 3)], rq[tri(1, 3)]);
    Rb[5 * 64 + lane] = pack8<T>(rq[tri(2, 3)], rq[tri(3, 3)]);
  }

  // ---- A blocks.  Off-diagonal (k < P), transposed: at(k, P) register i = A[16P + c][16k + 4g + i].
  // Diagonal, plain (row 16P + 4g + i, column 16P + c), stored as rows of N^T in LDS.
  f32x4 at[10];
#pragma unroll
  for (int P = 1; P < 4; ++P) {
    const float at_ = tak[16 * P + c16];
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const f32x4 bu = *(const f32x4*)(tbk + 16 * k + 4 * g);
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_exp2f(at_ - bu[i]) * gk[tri(k, P)][i];
      at[tri(k, P)] = v;
    }
  }
#pragma unroll
  for (int P = 0; P < 4; ++P) {
    const float bu = tbk[16 * P + c16];
    const f32x4 ar = *(const f32x4*)(tak + 16 * P + 4 * g);
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)  // (the exponent is discarded above the diagonal)
      v[i] = (c16 < 4 * g + i) ? __builtin_amdgcn_exp2f(ar[i] - bu) * gk[tri(P, P)][i] : 0.f;
    *(f32x4*)(nb + P * 256 + c16 * 16 + 4 * g) = v;  // N^T[c][4g + i] = N[4g + i][c]
  }
  wave_sync();

  // ---- T_PP = (I + N)^-1 by forward substitution: lane (g, c) solves column c of block g
  {
    const float* nt = nb + g * 256;
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = (r == c16) ? 1.f : 0.f;
#pragma unroll
    for (int j = 0; j < 15; ++j) {
      float n[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = *(const f32x4*)(nt + j * 16 + 4 * q);  // column j of N
#pragma unroll
        for (int e = 0; e < 4; ++e) n[4 * q + e] = v[e];
      }
#pragma unroll
      for (int r = j + 1; r < 16; ++r) x[r] = fmaf(-n[r], x[j], x[r]);
    }
    float* mt = mb + g * 256 + c16 * 16;  // T^T row c = column c of T
#pragma unroll
    for (int q = 0; q < 4; ++q) *(f32x4*)(mt + 4 * q) = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
  }
  wave_sync();
  f32x4 tpp[4], tppT[4];  // T_PP and T_PP^T in the accumulator layout
#pragma unroll
  for (int P = 0; P < 4; ++P) {
    tpp[P] = *(const f32x4*)(mb + P * 256 + c16 * 16 + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) tppT[P][i] = mb[P * 256 + (4 * g + i) * 16 + c16];
  }

  // ---- off-diagonal blocks, level L = P - S: T_PS = -T_PP Y_PS with Y_PS = sum_{k=S}^{P-1}
  // A_Pk T_kS, and (T^T)_SP = -Y_PS^T T_PP^T (left factors enter transposed: at, tppT, Y)
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  const f32x4 y10 = blk_mul(at[tri(0, 1)], tpp[0], z);
  const f32x4 y21 = blk_mul(at[tri(1, 2)], tpp[1], z);
  const f32x4 y32 = blk_mul(at[tri(2, 3)], tpp[2], z);
  const f32x4 t10 = -blk_mul(tppT[1], y10, z);
  const f32x4 t21 = -blk_mul(tppT[2], y21, z);
  const f32x4 tt01 = -blk_mul(y10, tppT[1], z);
  const f32x4 tt12 = -blk_mul(y21, tppT[2], z);
  const f32x4 tt23 = -blk_mul(y32, tppT[3], z);
  const f32x4 y20 = blk_mul(at[tri(1, 2)], t10, blk_mul(at[tri(0, 2)], tpp[0], z));
  const f32x4 y31 = blk_mul(at[tri(2, 3)], t21, blk_mul(at[tri(1, 3)], tpp[1], z));
  const f32x4 t20 = -blk_mul(tppT[2], y20, z);
  const f32x4 tt02 = -blk_mul(y20, tppT[2], z);
  const f32x4 tt13 = -blk_mul(y31, tppT[3], z);
  const f32x4 y30 =
      blk_mul(at[tri(2, 3)], t20, blk_mul(at[tri(1, 3)], t10, blk_mul(at[tri(0, 3)], tpp[0], z)));
  const f32x4 tt03 = -blk_mul(y30, tppT[3], z);

  // ---- T diag(beta), transposed blocks (S, P) scaled by beta on row 16S + 4g + i, written
  // as the scan's A fragments (fragment (P, j) = blocks (2j, P), (2j + 1, P))
  {
    f32x4 bs[4];
#pragma unroll
    for (int S = 0; S < 4; ++S) bs[S] = *(const f32x4*)(tbt + 16 * S + 4 * g);
    u32x4* Tb = (u32x4*)(rec + kGdn16Tb);
    Tb[0 * 64 + lane] = pack8<T>(tppT[0] * bs[0], z);
    Tb[1 * 64 + lane] = pack8<T>(tt01 * bs[0], tppT[1] * bs[1]);
    Tb[2 * 64 + lane] = pack8<T>(tt02 * bs[0], tt12 * bs[1]);
    Tb[3 * 64 + lane] = pack8<T>(tppT[2] * bs[2], z);
    Tb[4 * 64 + lane] = pack8<T>(tt03 * bs[0], tt13 * bs[1]);
    Tb[5 * 64 + lane] = pack8<T>(tt23 * bs[2], tppT[3] * bs[3]);
  }
}

// Chunk swizzle of the q rows in LDS (rows of CPR 16-byte chunks): logical chunk c of row r
// sits at c ^ f(r), so the 16 consecutive rows a B-fragment read touches (one chunk each)
// fall in distinct banks: f(r) = r mod 16 for 256-byte rows, (r / 2) mod 8 for 128-byte rows
// (two rows share one 256-byte bank line).  The k rows use lds_swizzle, which also keeps the
// transposing reads conflict-free.
template <int CPR>
__device__ __forceinline__ int rec_swizzle(int r) {
  static_assert(CPR == 8 || CPR == 16, "64- or 128-element rows");
  return CPR == 16 ? (r & 15) : ((r >> 1) & 7);
}

// Segment summaries (seg_mode 1) of the split recurrence: the state a segment leaves from a zero entry state (columns
// below D) and its transition matrix (columns from D, from the identity with v = 0).  Four waves of one workgroup, 16
// of its 64 columns each, one per SIMD; LDS holds one workgroup per CU, so the workgroup's columns set how many segments
// fill the device.  Bound by a wave's chain of products per chunk (its reads of the k rows and T fragments share the LDS
// with the other waves'): 1.4 us a chunk at D = 128 where two waves of 32 columns took 1.2, and twice the segments, so
// 20,000 tokens of 8 heads take summary + combine + replay 127 us, 157 with 32 columns.
template <typename T, int D>
__global__ void __launch_bounds__(256, 1) gdn_summary16_kernel(GdnArgs a) {
  constexpr int C = kChunk, KS = D / 32, ST = D / 16;
  constexpr int CPR = D / 8;                    // 16-byte chunks per k row
  constexpr int KB = C * D, VB = C * 64;        // elements of one slot's k rows, v slab
  constexpr int RB = kGdn16RecBytes;            // bytes of one slot's record
  constexpr int RPI = 64 / CPR;                 // k rows per copy instruction
  constexpr int NK = 16 / RPI;                  // copy instructions per wave for its 16 k rows
  constexpr int NREC = (RB / 1024 + 3) / 4;     // record blocks per wave (wave 3 repeats the last)
  constexpr int NDMA = NK + 2 + NREC;           // copies per wave per chunk
  static_assert(RB % 1024 == 0, "record of whole 1 KiB blocks");
  // three slots per array: chunk c lives in slot c % 3, so within the three-times unrolled
  // loop every slot offset is an instruction immediate
  __shared__ __attribute__((aligned(16))) T Ks[3 * KB];
  __shared__ __attribute__((aligned(16))) T Vs[3 * VB];
  __shared__ __attribute__((aligned(16))) char Rs[3 * RB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int bh = blockIdx.x, b = bh / a.H, hk = bh % a.H / a.G;
  const int vw = 64 * blockIdx.y;    // the workgroup's 64 state columns (>= D: the transition)
  const int v0 = vw + 16 * wave;     // this wave's 16
  const int seg = blockIdx.z;
  const int c_begin = seg * a.seg_len, c_end = min(a.NC, c_begin + a.seg_len);
  const bool trans = vw >= D;

  // ---- state: tile t, register i <-> row k = 32 (t/2) + 8g + 4 (t%2) + i, column v0 + c16
  f32x4 S[ST];
#pragma unroll
  for (int t = 0; t < ST; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kx = 32 * (t >> 1) + 8 * g + 4 * (t & 1) + i;
      S[t][i] = (trans && kx == v0 + c16 - D) ? 1.f : 0.f;
    }

  // ---- lane parts of the LDS addresses (elements; tile and slot offsets are immediates).
  // k rows use lds_swizzle, whose value for the rows a lane touches is fixed: A fragments
  // read row 16p + c16 (swizzle of c16), transposing reads row 32j + 4g + c16/4 (+16)
  // (swizzle 4 (c16/4) + g).
  const int ksw = lds_swizzle<CPR>(c16);
  int kAo[KS], kTo[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kAo[s] = c16 * D + 8 * ((4 * s + g) ^ ksw);
    // tile t = 2s (+1): lane supplies columns 32 s + 8 (c16 % 4) + 4 (t % 2) of row
    // 4g + c16/4 (+ 32j, + 16): chunk 4s + c16 % 4
    const int r0 = 4 * g + (c16 >> 2);
    kTo[s] = r0 * D + 8 * ((4 * s + (c16 & 3)) ^ lds_swizzle<CPR>(r0));
  }
  // v slab rows of 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 mod 8): the 16 rows a transposing read touches fall
  // in distinct banks
  const int vr0 = 4 * g + (c16 >> 2);
  const int vo = vr0 * 64 + 8 * ((2 * wave + ((c16 & 3) >> 1)) ^ ((vr0 >> 1) & 7)) + 4 * (c16 & 1);

  // ---- copies of chunk j into slot sl: wave w copies k and v slab rows 16w .. 16w + 15 (with their swizzles) and a
  // quarter of the record's 1 KiB blocks (wave 3 copies the last one again, so that every wave issues the same number of
  // copies).  Rows past T read as zeros.
  const uint32_t kst2 = (uint32_t)a.k_st * 2u, vst2 = (uint32_t)a.v_st * 2u;
  uint32_t kvo[NK], vvo[2];
#pragma unroll
  for (int r = 0; r < NK; ++r) {
    const int row = 16 * wave + RPI * r + lane / CPR, pc = lane % CPR;
    kvo[r] = row * kst2 + 16u * (pc ^ lds_swizzle<CPR>(row));
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int row = 16 * wave + 8 * r + lane / 8;
    vvo[r] = row * vst2 + 16u * ((lane % 8) ^ ((row >> 1) & 7));
  }
  const uint32_t rvo = 16u * lane;  // record blocks: the block offset is a scalar (always in range)
  const T* kb = (const T*)a.k + b * a.k_sb + hk * a.k_sh;
  const T* vb = (const T*)a.v + b * a.v_sb + hk * a.v_sh + (trans ? 0 : vw);
  const char* rb0 = (const char*)a.ws + (int64_t)bh * a.NC * RB;
  const int last = c_end - 1;
  // LDS byte offsets of this wave's copy destinations, in scalar registers
  const uint32_t mk = __builtin_amdgcn_readfirstlane(lds_offset(Ks + 16 * wave * D));
  const uint32_t mv = __builtin_amdgcn_readfirstlane(lds_offset(Vs + 16 * wave * 64));
  const uint32_t mr = __builtin_amdgcn_readfirstlane(lds_offset(Rs));
  auto copy_chunk = [&](int j, auto slot_c) {
    constexpr int sl = decltype(slot_c)::value;
    const int rows = min(a.T - j * C, C);
    const auto krs = buffer_rsrc(kb + (int64_t)j * C * a.k_st, (uint32_t)((rows - 1) * a.k_st + D) * 2u);
    // (transition columns take v = 0: an empty range, so that the copies only write zeros)
    const auto vrs = buffer_rsrc(vb + (int64_t)j * C * a.v_st, trans ? 0u : (uint32_t)((rows - 1) * a.v_st + 64) * 2u);
    const auto rrs = buffer_rsrc(rb0 + (int64_t)j * RB, RB);
#pragma unroll
    for (int r = 0; r < NK; ++r) dma_buf16_at(krs, kvo[r], 0, mk + (sl * KB + RPI * r * D) * 2);
#pragma unroll
    for (int r = 0; r < 2; ++r) dma_buf16_at(vrs, vvo[r], 0, mv + (sl * VB + 8 * r * 64) * 2);
#pragma unroll
    for (int r = 0; r < NREC; ++r) {
      const uint32_t blk = (uint32_t)min(NREC * wave + r, RB / 1024 - 1) * 1024u;
      dma_buf16_at(rrs, rvo, blk, mr + sl * RB + blk);
    }
  };

  auto body = [&](int c, auto slot_c) {
    constexpr int sl = decltype(slot_c)::value;
    // this wave's copies of chunk c have landed (only those of chunk c + 1 may be in
    // flight: loads complete in order), then the others'
    wait_vmcnt<NDMA>();
    __syncthreads();

    const T* Kl = Ks + sl * KB;
    const T* Vl = Vs + sl * VB;
    const char* Rl = Rs + sl * RB;
    const float* Fp = (const float*)(Rl + kGdn16F);
    const u32x4* Tb = (const u32x4*)(Rl + kGdn16Tb);

    // The LDS reads of each phase are issued before its first product and the scheduling
    // barriers keep that order (one wave per SIMD: no other wave hides a read's latency).
    // (1) reads: k rows as A fragments of K S (tile p: row 16p + c16), gC
    u32x4 kA[4][KS];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int s = 0; s < KS; ++s) kA[p][s] = lds16(Kl + 16 * p * D + kAo[s]);
    const float gC = Fp[192];
    __builtin_amdgcn_sched_barrier(0);

    // (2) K S with S as B fragments (k-step s: tiles 2s, 2s + 1); the same registers are the
    // A fragments of S^T; independent products adjacent, and S <- gC S issued between them
    // (a wave issues one instruction per cycle slot, so VALU work placed between products
    // runs while the matrix unit is busy)
    u32x4 sf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) sf[s] = pack8<T>(S[2 * s], S[2 * s + 1]);
    f32x4 ks[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) ks[p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int p = 0; p < 4; ++p) ks[p] = mfma16x16x32<T>(kA[p][s], sf[s], ks[p]);
#pragma unroll
    for (int t = 0; t < ST; ++t) S[t] *= gC;
    __builtin_amdgcn_sched_group_barrier(0x002, 2 * KS, 0);  // the S fragments
#pragma unroll
    for (int i = 0; i < 4 * KS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // chunk c + 2 goes to the slot chunk c - 1 used (every wave is past the barrier above);
    // issued here, behind the products, so the copies' issue does not delay them.  Past the
    // last chunk the copies repeat it, so every step issues the same count.
    copy_chunk(min(c + 2, last), std::integral_constant<int, (sl + 2) % 3>{});

    // (3) reads for X and U: v by transposing reads of the slab (lane c16 supplies row r0 + c16 / 4, columns
    // 16 wave + 4 (c16 % 4)) in the token slot order 32j + 4g + [0,4), 32j + 16 + 4g + [0,4), geik of the same tokens,
    // T diag(beta)
    u32x2 vlo[2], vhi[2];
    f32x4 wl[2], wh[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      vlo[j] = lds_read_tr16(Vl + 32 * j * 64 + vo);
      vhi[j] = lds_read_tr16(Vl + (32 * j + 16) * 64 + vo);
      wl[j] = *(const f32x4*)(Fp + 64 + 32 * j + 4 * g);
      wh[j] = *(const f32x4*)(Fp + 64 + 32 * j + 16 + 4 * g);
    }
    u32x4 tb[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) tb[f] = Tb[f * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);

    // (4) X = V - geik K S as B fragments over token steps j
    u32x4 xf[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x4 xl, xh;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xl[i] = elem16x2<T>(vlo[j], i) - wl[j][i] * ks[2 * j][i];
        xh[i] = elem16x2<T>(vhi[j], i) - wh[j][i] * ks[2 * j + 1][i];
      }
      xf[j] = pack8<T>(xl, xh);
    }
    __builtin_amdgcn_sched_barrier(0);

    // (5) reads for the state update: A fragments of K^T by
    // transposing reads (for tile t, lane c16 supplies row r0 + c16 / 4 and the 4 columns
    // 32 (t/2) + 8 (c16 % 4) + 4 (t%2) .., so lane r receives column 32 (t/2) + 8 (r/4) +
    // 4 (t%2) + r % 4, the state row of tile t); kf of the token slots
    u32x4 kT[2][ST];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < ST; ++t) {
        const T* pl = Kl + 32 * j * D + kTo[t >> 1] + 4 * (t & 1);
        const u32x2 lo = lds_read_tr16(pl);
        const u32x2 hi = lds_read_tr16(pl + 16 * D);
        kT[j][t] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    f32x4 kl[2], kh[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      kl[j] = *(const f32x4*)(Fp + 32 * j + 4 * g);
      kh[j] = *(const f32x4*)(Fp + 32 * j + 16 + 4 * g);
    }
    __builtin_amdgcn_sched_barrier(0);

    // (6) U = T diag(beta) X: tile P = tokens 16P + 4g + i (T is lower triangular); U as B fragments of the update in
    // the token slot order, weighted by kf
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    f32x4 U[4];
    U[0] = mfma16x16x32<T>(tb[0], xf[0], z);
    U[1] = mfma16x16x32<T>(tb[1], xf[0], z);
    U[2] = mfma16x16x32<T>(tb[2], xf[0], z);
    U[3] = mfma16x16x32<T>(tb[4], xf[0], z);
    U[2] = mfma16x16x32<T>(tb[3], xf[1], U[2]);
    U[3] = mfma16x16x32<T>(tb[5], xf[1], U[3]);
    u32x4 ukf[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      ukf[j] = pack8<T>(U[2 * j] * kl[j], U[2 * j + 1] * kh[j]);
    }

    // (7) S += K^T diag(kf) U
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < ST; ++t) S[t] = mfma16x16x32<T>(kT[j][t], ukf[j], S[t]);
  };

  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  copy_chunk(c_begin, S0{});
  copy_chunk(min(c_begin + 1, last), S1{});
  for (int c = c_begin; c < c_end; c += 3) {
    body(c, S0{});
    if (c + 1 < c_end) body(c + 1, S1{});
    if (c + 2 < c_end) body(c + 2, S2{});
  }

  float* sdst = a.seg_sum + ((int64_t)bh * (a.nseg - 1) + seg) * D * 2 * D;  // the exit state: [k][2D columns]
#pragma unroll
  for (int t = 0; t < ST; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kx = 32 * (t >> 1) + 8 * g + 4 * (t & 1) + i;
      sdst[kx * 2 * D + v0 + c16] = S[t][i];
    }
  // the copies issued past the last chunk land before the workgroup's LDS is released
  wait_vmcnt<0>();
}

// The scan with its output (seg_mode 0 and 2) on four waves: chain waves 0 and 1 run only
// the recurrence of their 16 columns (K S -> X -> U -> S update), and output waves 2 and 3
// compute the same columns' output rows and issue every copy.  A wave issues at most one
// instruction per cycle slot of its SIMD, and with one wave per SIMD the chain's step time
// is its instruction count; the output products, q reads, stores and copies move to the two
// SIMDs that the chain leaves idle.  Per chunk c, between the top barrier B0 and the
// middle barrier B1 the chain reads S_c's fragments from its registers and writes U_c's to
// LDS; after B1 it updates S and writes S_{c+1}'s fragments.  The output wave reads S_c's
// fragments before B1 (the chain overwrites them only after B1) and U_c's after B1 (the
// chain overwrites them only after the next B0).
template <typename T, int D, typename SEQ>
__global__ void __launch_bounds__(256, 1) gdn_scan16_pair_kernel(GdnArgs a, SEQ seqs) {
  constexpr int C = kChunk, KS = D / 32, ST = D / 16;
  constexpr int CPR = D / 8;                    // 16-byte chunks per k / q row
  constexpr int KB = C * D, VB = C * 32;        // elements of one slot's k (q) rows, v slab
  constexpr int RB = kGdn16RecBytes;            // bytes of one slot's record
  constexpr int RPI = 64 / CPR;                 // k / q rows per copy instruction
  constexpr int NKQ = 32 / RPI;                 // copy instructions per output wave for its 32 k (q) rows
  constexpr int NREC = (RB / 1024 + 1) / 2;     // record blocks per output wave (wave 3 repeats its last)
  constexpr int NDMA = 2 * NKQ + 2 + NREC;      // copies per output wave per chunk
  static_assert(RB % 1024 == 0, "record of whole 1 KiB blocks");
  __shared__ __attribute__((aligned(16))) T Ks[3 * KB];
  __shared__ __attribute__((aligned(16))) T Qs[3 * KB];
  __shared__ __attribute__((aligned(16))) T Vs[3 * VB];
  __shared__ __attribute__((aligned(16))) char Rs[3 * RB];
  __shared__ u32x4 SFs[2][KS][64];   // chain wave w: the state fragments at the current chunk's entry
  __shared__ u32x4 UFs[2][2][64];    // chain wave w: U fragments of the current chunk

  if (a.seg_mode != 2) gdn_signal_start(a);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool chain = wave < 2;
  const int pw = wave & 1;           // column half: chain wave pw and output wave 2 + pw share it
  const int g = lane >> 4, c16 = lane & 15;
  const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H, hk = h / a.G;
  const int vw = 32 * blockIdx.y;    // the workgroup's 32 state columns
  const int v0 = vw + 16 * pw;       // this wave pair's 16
  const int seg = blockIdx.z;
  const SeqView sq = gdn_seq(a, seqs, b);
  const int c_begin = std::is_same_v<SEQ, VarSeqs> ? 0 : seg * a.seg_len;
  const int c_end = std::is_same_v<SEQ, VarSeqs> ? sq.NC : min(a.NC, c_begin + a.seg_len);

  // the entry state: the call's; a replay's is segment 0's copy of it, or lies over the previous segment's summary
  const float* s0;
  int ld0 = D;
  if (a.seg_mode == 0) {
    s0 = gdn_state(a, a.s0, sq.row, h, D);
  } else if (seg == 0) {
    s0 = a.seg_in + (int64_t)bh * D * D;
  } else {
    s0 = a.seg_sum + ((int64_t)bh * (a.nseg - 1) + seg - 1) * D * 2 * D;
    ld0 = 2 * D;
  }

  // ---- chain: state tile t, register i <-> row k = 32 (t/2) + 8g + 4 (t%2) + i, column v0 + c16
  f32x4 S[ST];
  u32x4 sf[KS];
  if (chain) {
#pragma unroll
    for (int t = 0; t < ST; ++t) S[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (s0) {
#pragma unroll
      for (int t = 0; t < ST; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[t][i] = s0[(32 * (t >> 1) + 8 * g + 4 * (t & 1) + i) * ld0 + v0 + c16];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      sf[s] = pack8<T>(S[2 * s], S[2 * s + 1]);
      SFs[pw][s][lane] = sf[s];
    }
  }

  // ---- lane parts of the LDS addresses (elements; tile and slot offsets are immediates),
  // as in gdn_summary16_kernel
  const int ksw = lds_swizzle<CPR>(c16);
  int kAo[KS], qBo[KS], kTo[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kAo[s] = c16 * D + 8 * ((4 * s + g) ^ ksw);
    qBo[s] = c16 * D + 8 * ((4 * s + g) ^ rec_swizzle<CPR>(c16));
    const int r0 = 4 * g + (c16 >> 2);
    kTo[s] = r0 * D + 8 * ((4 * s + (c16 & 3)) ^ lds_swizzle<CPR>(r0));
  }
  const int vo = (4 * g + (c16 >> 2)) * 32 + 16 * pw + 4 * (c16 & 3);

  // ---- copies (output waves): wave 2 + w copies k and q rows 32w .. 32w + 31, v slab rows
  // 32w .. 32w + 31 and half of the record's 1 KiB blocks (wave 3 copies its last block
  // twice when the count is odd).  Rows past T read as zeros.
  const int cw = wave & 1;
  const uint32_t kst2 = (uint32_t)a.k_st * 2u, qst2 = (uint32_t)a.q_st * 2u, vst2 = (uint32_t)a.v_st * 2u;
  uint32_t kvo[NKQ], qvo[NKQ], vvo[2];
#pragma unroll
  for (int r = 0; r < NKQ; ++r) {
    const int row = 32 * cw + RPI * r + lane / CPR, pc = lane % CPR;
    kvo[r] = row * kst2 + 16u * (pc ^ lds_swizzle<CPR>(row));
    qvo[r] = row * qst2 + 16u * (pc ^ rec_swizzle<CPR>(row));
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) vvo[r] = (32 * cw + 16 * r + lane / 4) * vst2 + 16u * (lane % 4);
  const uint32_t rvo = 16u * lane;
  const T* kb = (const T*)a.k + sq.ko + hk * a.k_sh;
  const T* qb = (const T*)a.q + sq.qo + h * a.q_sh;
  const T* vb = (const T*)a.v + sq.vo + hk * a.v_sh + vw;
  const char* rb0 = (const char*)a.ws + (sq.chunk0 * a.H + (int64_t)h * sq.NC) * RB;
  const int last = c_end - 1;
  const uint32_t mk = __builtin_amdgcn_readfirstlane(lds_offset(Ks + 32 * cw * D));
  const uint32_t mq = __builtin_amdgcn_readfirstlane(lds_offset(Qs + 32 * cw * D));
  const uint32_t mv = __builtin_amdgcn_readfirstlane(lds_offset(Vs + 32 * cw * 32));
  const uint32_t mr = __builtin_amdgcn_readfirstlane(lds_offset(Rs));
  auto copy_chunk = [&](int j, auto slot_c) {
    constexpr int sl = decltype(slot_c)::value;
    const int rows = min(sq.T - j * C, C);
    const auto krs = buffer_rsrc(kb + (int64_t)j * C * a.k_st, (uint32_t)((rows - 1) * a.k_st + D) * 2u);
    const auto qrs = buffer_rsrc(qb + (int64_t)j * C * a.q_st, (uint32_t)((rows - 1) * a.q_st + D) * 2u);
    const auto vrs = buffer_rsrc(vb + (int64_t)j * C * a.v_st, (uint32_t)((rows - 1) * a.v_st + 32) * 2u);
    const auto rrs = buffer_rsrc(rb0 + (int64_t)j * RB, RB);
#pragma unroll
    for (int r = 0; r < NKQ; ++r) {
      dma_buf16_at(krs, kvo[r], 0, mk + (sl * KB + RPI * r * D) * 2);
      dma_buf16_at(qrs, qvo[r], 0, mq + (sl * KB + RPI * r * D) * 2);
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) dma_buf16_at(vrs, vvo[r], 0, mv + (sl * VB + 16 * r * 32) * 2);
#pragma unroll
    for (int r = 0; r < NREC; ++r) {
      const uint32_t blk = (uint32_t)min(NREC * cw + r, RB / 1024 - 1) * 1024u;
      dma_buf16_at(rrs, rvo, blk, mr + sl * RB + blk);
    }
  };

  const auto orsrc = buffer_rsrc((const T*)a.o + sq.tok0 * a.H * D, (uint32_t)((int64_t)sq.T * a.H * D * 2));
  const uint32_t oo = (uint32_t)((c16 * a.H + h) * D + v0 + 4 * g) * 2u;
  const uint32_t otok = (uint32_t)a.H * D * 2u;
  f32x4 o[4];

  auto body = [&](int c, auto slot_c) {
    constexpr int sl = decltype(slot_c)::value;
    // B0: the output waves' copies of chunk c have landed (only chunk c + 1's and the
    // previous chunk's stores may be in flight; loads complete in order), the chain's S_c
    // fragments are written
    wait_vmcnt<NDMA>();
    __syncthreads();
    const T* Kl = Ks + sl * KB;
    const T* Ql = Qs + sl * KB;
    const T* Vl = Vs + sl * VB;
    const char* Rl = Rs + sl * RB;
    const float* Fp = (const float*)(Rl + kGdn16F);
    const u32x4* Tb = (const u32x4*)(Rl + kGdn16Tb);
    const u32x4* Rb = (const u32x4*)(Rl + kGdn16Rb);
    f32x4 ks[4];
    u32x4 ukf[2], kT[2][ST];
    if (chain) {
      // (1) gC, then the k rows as A fragments of K S (tile p: row 16p + c16); LDS reads
      // return in order, so the first product waits for gC and its own two fragments only
      const float gC = Fp[192];
      u32x4 kA[4][KS];
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int s = 0; s < KS; ++s) kA[p][s] = lds16(Kl + 16 * p * D + kAo[s]);
      __builtin_amdgcn_sched_barrier(0);
      // (2) K S (S_c as B fragments) with S <- gC S and the reads X and U need (v by
      // transposing reads of the slab in the token slot order, geik, kf, T diag(beta))
      // issued between the products
#pragma unroll
      for (int p = 0; p < 4; ++p) ks[p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int p = 0; p < 4; ++p) ks[p] = mfma16x16x32<T>(kA[p][s], sf[s], ks[p]);
#pragma unroll
      for (int t = 0; t < ST; ++t) S[t] *= gC;
      u32x2 vlo[2], vhi[2];
      f32x4 wl[2], wh[2], kl[2], kh[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        vlo[j] = lds_read_tr16(Vl + 32 * j * 32 + vo);
        vhi[j] = lds_read_tr16(Vl + (32 * j + 16) * 32 + vo);
        wl[j] = *(const f32x4*)(Fp + 64 + 32 * j + 4 * g);
        wh[j] = *(const f32x4*)(Fp + 64 + 32 * j + 16 + 4 * g);
      }
      u32x4 tb[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) tb[f] = Tb[f * 64 + lane];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        kl[j] = *(const f32x4*)(Fp + 32 * j + 4 * g);
        kh[j] = *(const f32x4*)(Fp + 32 * j + 16 + 4 * g);
      }
#pragma unroll
      for (int i = 0; i < 4 * KS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two decay multiplies
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // a read
      }
      __builtin_amdgcn_sched_barrier(0);
      // (3) K^T's A fragments of the update by transposing reads, issued under X and U (for
      // tile t, lane c16 supplies row r0 + c16 / 4 and the 4 columns 32 (t/2) + 8 (c16 % 4)
      // + 4 (t%2) .., so lane r receives the state row of tile t)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < ST; ++t) {
          const T* pl = Kl + 32 * j * D + kTo[t >> 1] + 4 * (t & 1);
          const u32x2 lo = lds_read_tr16(pl);
          const u32x2 hi = lds_read_tr16(pl + 16 * D);
          kT[j][t] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
      // (4) X = V - geik K S as B fragments over token steps j
      u32x4 xf[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x4 xl, xh;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          xl[i] = elem16x2<T>(vlo[j], i) - wl[j][i] * ks[2 * j][i];
          xh[i] = elem16x2<T>(vhi[j], i) - wh[j][i] * ks[2 * j + 1][i];
        }
        xf[j] = pack8<T>(xl, xh);
      }
      // (6) U = T diag(beta) X (tile P = tokens 16P + 4g + i), plain for the output wave and
      // weighted by kf for the update
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      f32x4 U[4];
      U[0] = mfma16x16x32<T>(tb[0], xf[0], z);
      U[1] = mfma16x16x32<T>(tb[1], xf[0], z);
      U[2] = mfma16x16x32<T>(tb[2], xf[0], z);
      U[3] = mfma16x16x32<T>(tb[4], xf[0], z);
      U[2] = mfma16x16x32<T>(tb[3], xf[1], U[2]);
      U[3] = mfma16x16x32<T>(tb[5], xf[1], U[3]);
#pragma unroll
      for (int i = 0; i < 2 * ST; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);  // two transposing reads
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 1);  // X
      }
#pragma unroll
      for (int i = 0; i < 6; ++i) __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        UFs[pw][j][lane] = pack8<T>(U[2 * j], U[2 * j + 1]);
        ukf[j] = pack8<T>(U[2 * j] * kl[j], U[2 * j + 1] * kh[j]);
      }
    } else {
      // chunk c + 2 goes to the slot chunk c - 1 used (every wave is past B0); past the last
      // chunk the copies repeat it, so every step issues the same count
      copy_chunk(min(c + 2, last), std::integral_constant<int, (sl + 2) % 3>{});
      // q rows as B fragments of S^T Q^T (tile p': row 16p' + c16), S_c's fragments from the
      // chain partner; O^T tile p' (rows = columns v0 + 4g + i, cols = tokens 16p' + c16)
      u32x4 qB[4][KS];
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int s = 0; s < KS; ++s) qB[p][s] = lds16(Ql + 16 * p * D + qBo[s]);
#pragma unroll
      for (int s = 0; s < KS; ++s) sf[s] = SFs[pw][s][lane];
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) o[pp] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int pp = 0; pp < 4; ++pp) o[pp] = mfma16x16x32<T>(sf[s], qB[pp][s], o[pp]);
    }
    // B1: U_c's fragments are written; every read of S_c's is done
    __syncthreads();
    if (chain) {
      // (7) S += K^T diag(kf) U, then S_{c+1}'s fragments
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < ST; ++t) S[t] = mfma16x16x32<T>(kT[j][t], ukf[j], S[t]);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        sf[s] = pack8<T>(S[2 * s], S[2 * s + 1]);
        SFs[pw][s][lane] = sf[s];
      }
    } else {
      // output, second term: + U^T Rq^T, scaled first term by geqs of the token; 8-byte
      // row pieces O[token][v0 + 4g ..] (the whole offset in the lane's voffset: only that
      // part is range-checked, rows past T are dropped)
      u32x4 uf[2], rq[6];
#pragma unroll
      for (int j = 0; j < 2; ++j) uf[j] = UFs[pw][j][lane];
#pragma unroll
      for (int f = 0; f < 6; ++f) rq[f] = Rb[f * 64 + lane];
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) {
        f32x4 x = o[pp] * Fp[128 + 16 * pp + c16];
        if (pp < 2) {
          x = mfma16x16x32<T>(uf[0], rq[pp], x);
        } else {
          x = mfma16x16x32<T>(uf[0], rq[2 * pp - 2], x);
          x = mfma16x16x32<T>(uf[1], rq[2 * pp - 1], x);
        }
        const u32x2 pk = {pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3])};
        __builtin_amdgcn_raw_buffer_store_b64(pk, orsrc, oo + (uint32_t)(c * C + 16 * pp) * otok, 0, 0);
      }
    }
  };

  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  if (!chain) {
    copy_chunk(c_begin, S0{});
    copy_chunk(min(c_begin + 1, last), S1{});
  }
  for (int c = c_begin; c < c_end; c += 3) {
    body(c, S0{});
    if (c + 1 < c_end) body(c + 1, S1{});
    if (c + 2 < c_end) body(c + 2, S2{});
  }

  float* sdst = chain && seg == a.nseg - 1 ? gdn_state(a, a.s_out, sq.row, h, D) : nullptr;
  if (sdst) {
#pragma unroll
    for (int t = 0; t < ST; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kx = 32 * (t >> 1) + 8 * g + 4 * (t & 1) + i;
        sdst[kx * D + v0 + c16] = S[t][i];
      }
  }
  // the copies issued past the last chunk land before the workgroup's LDS is released
  wait_vmcnt<0>();
}

// Entry states of the segments from their summaries (fp32): E_0 = s0 (or 0) and E_s = M_{s-1} E_{s-1} + B_{s-1}, where
// summary s - 1 holds [B | M] row by row.  E_s goes over B_{s-1}, whose columns only this workgroup reads.
// One workgroup of four waves per (sequence-head, 16 state columns), a wave D / 4 rows of the product on
// v_mfma_f32_16x16x4f32 with the k index permuted (step 4 j + e contracts k = 16 j + 4 g + e), so that the four lanes
// of a row load 64 consecutive bytes of M.  The chain is one product per segment: M and B are loaded two segments ahead, and the state
// passes between the waves through LDS.  Bound by latency, about 2.8 us a segment (its D / 8 dependent products take 1):
// 20,000 tokens of 8 heads in 5 segments 13.8 us, 85 us with the products on VALU and M staged through LDS.
template <int D>
__global__ void __launch_bounds__(256) gdn_seg_combine_kernel(GdnArgs a) {
  constexpr int RT = D / 64, KL = D / 4;  // 16-row tiles per wave; k values per lane
  __shared__ __attribute__((aligned(16))) float cur[2][16][D + 4];  // the entry state's columns, [column][row]
  const int bh = blockIdx.x, j0 = 16 * blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const float* s0 = gdn_state(a, a.s0, bh / a.H, bh % a.H, D);
  f32x4 S[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * (RT * wave + t) + 4 * g + i;
      S[t][i] = s0 ? s0[row * D + j0 + c] : 0.f;
    }
  f32x4 m[2][RT][KL / 4], B[2][RT];  // of summary sg in slot sg % 2, loaded two steps ahead
  auto load = [&](int sg, auto slot_c) {
    constexpr int sl = decltype(slot_c)::value;
    const float* sum = a.seg_sum + ((int64_t)bh * (a.nseg - 1) + sg) * D * 2 * D;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const float* mr = sum + (16 * (RT * wave + t) + c) * 2 * D + D + 4 * g;
#pragma unroll
      for (int i = 0; i < KL / 4; ++i) m[sl][t][i] = *(const f32x4*)(mr + 16 * i);
#pragma unroll
      for (int i = 0; i < 4; ++i) B[sl][t][i] = sum[(16 * (RT * wave + t) + 4 * g + i) * 2 * D + j0 + c];
    }
  };
  auto step = [&](int sg, auto slot_c) {
    constexpr int sl = decltype(slot_c)::value;
    float* in = j0 + c + (sg ? a.seg_sum + ((int64_t)bh * (a.nseg - 1) + sg - 1) * D * 2 * D : a.seg_in + (int64_t)bh * D * D);
    const int ld = sg ? 2 * D : D;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int r0 = 16 * (RT * wave + t) + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) in[(r0 + i) * ld] = S[t][i];
      *(f32x4*)&cur[sl][c][r0] = S[t];
    }
    if (sg + 1 == a.nseg) return;
    __syncthreads();  // (the other buffer's readers are past the previous step's barrier)
    f32x4 acc[RT][2];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      acc[t][0] = B[sl][t];
      acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < KL / 4; ++i) {
      const f32x4 v = *(const f32x4*)&cur[sl][c][16 * i + 4 * g];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          acc[t][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[sl][t][i][e], v[e], acc[t][e & 1], 0, 0, 0);
    }
    if (sg + 3 < a.nseg) load(sg + 2, slot_c);
#pragma unroll
    for (int t = 0; t < RT; ++t) S[t] = acc[t][0] + acc[t][1];
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  load(0, S0{});
  if (a.nseg > 2) load(1, S1{});
  for (int sg = 0; sg < a.nseg; sg += 2) {
    step(sg, S0{});
    if (sg + 1 < a.nseg) step(sg + 1, S1{});
  }
}

// Segment count and length of a launch (nseg = 1: the plain scan); no segment is empty.
// The plan assumes MI355X's 256 compute units rather than querying the device, so the
// plan of a given shape and schedule does not depend on the GPU (or partition).  The
// schedule does: a launch with a start flag (the overlapped prefill, which a caller picks
// from the device's CU count and never under graph capture or autograd) takes the plain
// scan, and the plain and segmented scans differ in rounding only (the segment entry
// states are combined in fp32; agreement at 1e-2 of the output is tested at T = 65,536).
static int64_t gdn16_plan(int64_t BH, int NC, int D, int& nseg, int& seg_len) {
  int64_t states;  // of scratch per sequence-head
  nseg = gdn16_segments(BH, NC, D, 256, states);
  seg_len = (NC + nseg - 1) / nseg;
  nseg = (NC + seg_len - 1) / seg_len;
  return states;
}

size_t gdn16_workspace_bytes(int64_t BH, int64_t NC, int D) {
  int nseg, seg_len;
  const int64_t states = gdn16_plan(BH, (int)NC, D, nseg, seg_len);
  return (size_t)(BH * NC) * (size_t)kGdn16RecBytes + (size_t)(BH * states * D * D) * sizeof(float);
}

template <typename T, int D>
static int launch16(const GdnArgs& a0, hipStream_t s) {
  GdnArgs a = a0;
  const int64_t BH = (int64_t)a.B * a.H, items = (int64_t)a.NC * BH;
  gdn_prep16_kernel<T, D, DenseSeqs><<<dim3((unsigned)((items + 3) / 4)), dim3(256), 0, s>>>(a, {});
  int rc = check_launch("chunk_gated_delta_rule(prep16)");
  if (rc) return rc;
  gdn16_plan(BH, a.NC, D, a.nseg, a.seg_len);
  // with a start flag the caller runs another kernel beside the recurrence (the overlapped
  // prefill): the plain scan's few workgroups then run beside it, where the segment passes
  // would take every CU first
  if (a.start_flag) {
    a.nseg = 1;
    a.seg_len = a.NC;
  }
  if (a.nseg == 1) {
    a.seg_mode = 0;
    gdn_scan16_pair_kernel<T, D, DenseSeqs><<<dim3((unsigned)BH, D / 32, 1), dim3(256), 0, s>>>(a, {});
    return check_launch("chunk_gated_delta_rule(scan16)");
  }
  // long sequences with few heads: segment summaries, their entry states, then the replays
  a.seg_sum = (float*)((char*)a.ws + (size_t)items * kGdn16RecBytes);
  a.seg_in = a.seg_sum + BH * (a.nseg - 1) * D * 2 * D;
  a.seg_mode = 1;
  gdn_summary16_kernel<T, D><<<dim3((unsigned)BH, 2 * D / 64, a.nseg - 1), dim3(256), 0, s>>>(a);
  rc = check_launch("chunk_gated_delta_rule(summary16)");
  if (rc) return rc;
  gdn_seg_combine_kernel<D><<<dim3((unsigned)BH, D / 16), dim3(256), 0, s>>>(a);
  rc = check_launch("chunk_gated_delta_rule(combine16)");
  if (rc) return rc;
  a.seg_mode = 2;
  gdn_scan16_pair_kernel<T, D, DenseSeqs><<<dim3((unsigned)BH, D / 32, a.nseg), dim3(256), 0, s>>>(a, {});
  return check_launch("chunk_gated_delta_rule(replay16)");
}

// Ragged sequences packed along tokens: the plain scan of all of them in one launch each (a batch of prompts has heads
// enough to fill the device; the longest sequence's chunks set the time).  12 prompts of 64 .. 2,048 tokens, 8 heads: prep
// 22 and scan 48 us; one by one 157 and 187 with 43 + 35 for the split ones, and a gather and a scatter of the state each.
template <typename T, int D>
static int launch16_var(const GdnArgs& a0, const VarSeqs& v, hipStream_t s) {
  GdnArgs a = a0;
  a.nseg = 1;
  a.seg_mode = 0;
  const int64_t items = (int64_t)(v.chunk0[v.n - 1] + (v.len[v.n - 1] + 63) / 64) * a.H;
  gdn_prep16_kernel<T, D, VarSeqs><<<dim3((unsigned)((items + 3) / 4)), dim3(256), 0, s>>>(a, v);
  const int rc = check_launch("gated_delta_prefill(prep16)");
  if (rc) return rc;
  gdn_scan16_pair_kernel<T, D, VarSeqs><<<dim3((unsigned)(v.n * a.H), D / 32, 1), dim3(256), 0, s>>>(a, v);
  return check_launch("gated_delta_prefill(scan16)");
}

template <typename T>
static int launch16_d(const GdnArgs& a, const VarSeqs* v, int D, hipStream_t s) {
  if (v) return D == 128 ? launch16_var<T, 128>(a, *v, s) : launch16_var<T, 64>(a, *v, s);
  return D == 128 ? launch16<T, 128>(a, s) : launch16<T, 64>(a, s);
}

int launch_gdn16(const GdnArgs& a, const VarSeqs* v, int dtype, int D, hipStream_t s) {
  return dtype == ATMA_BF16 ? launch16_d<bf16>(a, v, D, s) : launch16_d<f16>(a, v, D, s);
}

}  // namespace atma
