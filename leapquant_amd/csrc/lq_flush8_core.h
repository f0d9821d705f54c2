// Per-head flush of GDN 128 x 128 heads at ranks 5 to 8 (the rank ablation, /root/reference/leapquant/kernels.py:1091,
// 1123, 1744-1772), shared by the standalone flush and the one-launch decode: the four-wave layout of lq_flush_core.h with
// eight factor columns, so that four heads share a CU.  The factor products carry the columns as the MFMA rows 4 q + i
// mod 8 (lane group q): the A operands' rows 8 .. 15 repeat rows 0 .. 7, so lane groups 0, 1 hold columns 0 .. 3, 4 .. 7
// for one channel group and lane groups 2, 3 for the other.
//
// CholeskyQR of these ranks drops a column whose pivot has lost all but 1e-6 of its Gram diagonal (1 / L_jj = 0) instead
// of flooring the pivot; columns past R are zero and stay zero.  Gram, factor and substitution run in fp64: a column that
// depends on the earlier ones leaves a pivot of ~1e-14 G_jj in fp64, but fp32 sums of 128 rows leave ~1e-6 G_jj of
// rounding -- the drop threshold itself -- so in fp32 whether such a column is dropped would be up to the rounding.
#pragma once
#include "lq_flush_core.h"

namespace {
namespace lqf {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int R8 = 8, TRI8 = R8 * (R8 + 1) / 2;   // factor columns; entries of a packed lower triangle, (r, c) at r (r + 1) / 2 + c

__device__ __forceinline__ f16_t half_bits(_Float16 x) { return __builtin_bit_cast(f16_t, x); }

struct FlushShared8 {
  static constexpr bool conflict_free = true;
  union {
    bf16_t op[3][KD][OPS4];      // rebuild operands of one window half [c or v][j]
    struct {                     // after the rebuild
      union {
        f32x4 qpart[2 * NW4][VD]; // partial Q rows of 16 channels each, four columns at a time
        struct {                 // CholeskyQR
          double gp[NW4][TRI8];  // per-wave partial Gram
          double lf[TRI8];       // its factor L; 1 / L_jj on the diagonal
          double col[R8];        // one column of L (wave 0's exchange)
        };
        float rmx[4 * NW4][VD + RMP];   // per-(wave, lane group) row maxima of the scaled residual
      };
      float rq[VD];              // qmax / row scale
      f16_t ppT[R8][KD + FTP];   // P16^T, then U16^T
      f16_t uoT[R8][KD + FTP];   // old U^T, fp16 (MFMA operand)
      f16_t qoT[R8][VD + FTP];   // old Q^T, fp16
      f16x4 qn16[2][VD];         // Q16 rows [v][r] (residual B operand)
      f32x4 mb[NW4][R8][2];      // per-wave broadcast of an 8 x 8 product: [r][a]
      f32x4 qv[2][VD];           // Q rows, fp32
    } r;
  };
  float skl[KD];                 // column factor of the dequant (Sk)
  float svr[VD];                 // row factor of the dequant (Sv pn / qmax)
  float w[LPMAX];
  f16x4 uo16[2][KD];             // old U rows [c][a], a >= R zero
  f16x4 qo16[2][VD];             // old Q rows [v][a], a >= R zero
  f16_t qT[R8][VD + FTP];        // Q^T operand of the P steps: fp16-rounded Q0, then Q16
  unsigned long long due;        // persistent flush: the workgroup's next candidate
};
static_assert(sizeof(FlushShared8) <= 40960, "four workgroups per CU: 160 KiB of LDS");

// M[a][4 b + i] = sum_k X[k][a] Y[k][4 b + i], a < 8, for this lane's block b, from the fp16 transposed operands X^T, Y^T
// ([8][128 (+ pad)]): the lanes l16 < 8 of groups 0, 1 hold M[4 q + i][l16] and share it through the wave's LDS words
__device__ __forceinline__ void gram8(FlushShared8& sh, const f16_t (*XT)[128 + FTP], const f16_t (*YT)[128 + FTP], int b,
                                      float (&M)[R8][4]) {
  const int l = lane4(), q = l >> 4, l16 = l & 15;
  f32x4 macc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    macc = mma32(*(const f16x8*)&XT[l16 & 7][32 * ks + 8 * q], *(const f16x8*)&YT[l16 & 7][32 * ks + 8 * q], macc);
  f32x4 (*mb)[2] = sh.r.mb[wave4()];
  if (l16 < R8 && q < 2) mb[l16][q] = macc;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 x = mb[4 * b + i][h];
#pragma unroll
      for (int a = 0; a < 4; ++a) M[4 * h + a][i] = x[a];
    }
}
// s[i] = sum_a x[a] M[a][i] over the row x of an fp16 factor (both blocks)
__device__ __forceinline__ f32x4 row_times(const f16x4 x0, const f16x4 x1, const float (&M)[R8][4]) {
  const f32x4 a = from_h4(x0), b = from_h4(x1);
  f32x4 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float c = a[0] * M[0][i];
#pragma unroll
    for (int k = 1; k < 4; ++k) c += a[k] * M[k][i];
#pragma unroll
    for (int k = 0; k < 4; ++k) c += b[k] * M[4 + k][i];
    s[i] = c;
  }
  return s;
}
// P = B^T Q + pn U_old (Q_old^T Q) for the wave's two channel groups, fp16-rounded (kernels.py:1580-1700), as p_step4: lane
// (q, l16) returns P[32 w + 16 g + l16][4 b .. 4 b + 3], g = q >> 1, b = q & 1 (zero for columns >= R).  TR: forms the
// transposed blocks of B into bt (one exact MFMA each against the identity).
template <bool TR>
__device__ __forceinline__ f32x4 p_step8(FlushShared8& sh, const f16x4 (&bh)[2][8], f16x4 (&bt)[2][8], float pn, int R) {
  const int l = lane4(), w = wave4(), q = l >> 4, l16 = l & 15, b = q & 1;
  const bool g1 = q >= 2;
  float M[R8][4];
  gram8(sh, sh.r.qoT, sh.qT, b, M);
  const int c = 32 * w + (g1 ? 16 : 0) + l16;
  const f32x4 corr = row_times(sh.uo16[0][c], sh.uo16[1][c], M);
  f16x4 ident;
#pragma unroll
  for (int i = 0; i < 4; ++i) ident[i] = (4 * q + i == l16) ? (_Float16)1.0f : (_Float16)0.0f;
  f32x4 pacc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int nt = 0; nt < 8; ++nt) {                    // P^T[r][c] = sum_v Q^T[r][v] B[c][v] (k = v)
    const f16x4 aq = *(const f16x4*)&sh.qT[l16 & 7][16 * nt + 4 * q];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      if constexpr (TR) bt[g][nt] = pinned(to_h4(mma16(bh[g][nt], ident, f32x4{0.f, 0.f, 0.f, 0.f})));
      pacc[g] = mma16(aq, bt[g][nt], pacc[g]);
    }
  }
  f32x4 p;
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] = 4 * b + i < R ? hround((g1 ? pacc[1][i] : pacc[0][i]) + pn * corr[i]) : 0.f;
  return p;
}

// 1 / sqrt(x) in fp64 from the hardware's estimate, two Newton steps
__device__ __forceinline__ double rsq_d(double x) {
  double y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int k = 0; k < 2; ++k) y = fma(y * 0.5, fma(-x * y, y, 1.0), y);
  return y;
}
// One CholeskyQR pass on the rows sh.r.qv (kernels.py:1744-1772).  The Gram by fp64 MFMA (v_mfma_f64_16x16x4: lane (q, l16)
// holds A[l16][q], B[q][l16] and rows q + 4 i of D), each wave over its 32 rows, one multiplication of a register with
// itself per four rows; the factor on wave 0, right-looking, one triangle entry per lane; the substitution one row per
// thread of waves 0 and 1.  `put(v, x0, x1)` takes each row's result.  (An eight-wave layout at two heads per CU, with the
// Gram as 36 wave reductions and the triangle gathered by readlane on one wave, took 600 us for 8192 due heads at W = 64
// and 562 at W = 16; this one 307 and 237.  Bound, as the four-wave flush at R <= 4 (158 and 134 us), by VALU issue.)
template <class F>
__device__ __forceinline__ void cholqr8_pass(FlushShared8& sh, F put) {
  const int tid = tid4(), l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), q = l >> 4, l16 = l & 15;
  {
    f64x4 g = {0.0, 0.0, 0.0, 0.0};
    const float* X = (const float*)sh.r.qv[(l16 >> 2) & 1] + (l16 & 3);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const float xf = X[4 * (32 * w + 4 * s + q)];
      const double x = l16 < R8 ? (double)xf : 0.0;
      g = __builtin_amdgcn_mfma_f64_16x16x4f64(x, x, g, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = q + 4 * i;
      if (l16 <= r) sh.r.gp[w][r * (r + 1) / 2 + l16] = g[i];
    }
  }
  __syncthreads();
  if (w == 0) {
    __builtin_amdgcn_s_setprio(3);
    const int t = l < TRI8 ? l : 0;
    int r = 0;                                        // entry (r, c) of lane t
#pragma unroll
    for (int k = 1; k < R8; ++k) r += t >= k * (k + 1) / 2 ? 1 : 0;
    const int c = t - r * (r + 1) / 2;
    const double g0 = ((sh.r.gp[0][t] + sh.r.gp[1][t]) + sh.r.gp[2][t]) + sh.r.gp[3][t];
    double a = g0;
#pragma unroll
    for (int j = 0; j < R8; ++j) {
      const int tj = j * (j + 1) / 2 + j;
      const double gjj = rl_d(g0, tj), d = rl_d(a, tj);
      const double inv = d > 1e-6 * gjj + 1e-30 ? rsq_d(fmax(d, 1e-30)) : 0.0;
      if (c == j) a = r == j ? inv : a * inv;         // column j of L
      if (j + 1 < R8) {
        if (c == j) sh.r.col[r] = a;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const double lr = sh.r.col[r], lc = sh.r.col[c];
        if (c > j) a = fma(-lr, lc, a);
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (l < TRI8) sh.r.lf[t] = a;
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();
  if (tid < VD) {
    const int v = tid;
    const f32x4 p0 = sh.r.qv[0][v], p1 = sh.r.qv[1][v];
    double x[R8];
    float y[R8];
#pragma unroll
    for (int j = 0; j < R8; ++j) {
      double ac = j < 4 ? (double)p0[j & 3] : (double)p1[j & 3];
#pragma unroll
      for (int m = 0; m < j; ++m) ac = fma(-x[m], sh.r.lf[j * (j + 1) / 2 + m], ac);
      x[j] = ac * sh.r.lf[j * (j + 1) / 2 + j];
      y[j] = (float)x[j];
    }
    put(v, f32x4{y[0], y[1], y[2], y[3]}, f32x4{y[4], y[5], y[6], y[7]});
  }
  __syncthreads();
}

__device__ void flush_head8(FlushShared8& sh, const lq_state& st, const float* __restrict__ Q0, int slot, int hv,
                            float qmax, int* sched = nullptr) {
  const int HV = st.HV, L = st.L, R = st.R;
  const long long sh_ = (long long)slot * HV + hv;
  const int tid = tid4(), l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), q = l >> 4, l16 = l & 15;
  char* base = block_base(st, slot, hv);
  const float* Sk = (const float*)(base + VD * KD);
  const float* Sv = Sk + KD;
  f16_t* UQ = (f16_t*)(base + VD * KD + 4 * (KD + VD));
  const bool two = L > HALF;                          // window halves

  // ---- stage 1: every load of the head up front ----
  const float pn = fmaxf(st.Pbuf[sh_], LQ_PNMIN);     // kernels.py:1471
  const float rpn = 1.0f / pn;                        // kernels.py:1477
  const int cv = tid & 127;                           // column (tid < 128) or row of the stage-1 loads
  const bool colt = tid < KD;
  const float scv = colt ? Sk[cv] : Sv[cv];
  f16_t uqv[R8];
  float q0v[R8];
#pragma unroll
  for (int a = 0; a < R8; ++a) {
    uqv[a] = UQ[min(a, R - 1) * (KD + VD) + (colt ? 0 : KD) + cv];
    q0v[a] = Q0[cv * R + min(a, R - 1)];
  }
  const float wv = st.Wbuf[sh_ * L + min(tid, L - 1)];
  WinHalf win;
  load_half<KD, VD>(win, st, slot, hv, L, 0);
  uint32_t wds[2][8];                                 // loaded after the first window half's products
  {
    f16x4 f[2];
#pragma unroll
    for (int a = 0; a < R8; ++a) f[a >> 2][a & 3] = __builtin_bit_cast(_Float16, a < R ? uqv[a] : (f16_t)0);
    if (colt) {
      sh.skl[cv] = scv;
      sh.uo16[0][cv] = f[0];
      sh.uo16[1][cv] = f[1];
    } else {
      sh.svr[cv] = scv * (pn / qmax);                                                 // kernels.py:1483
      sh.qo16[0][cv] = f[0];
      sh.qo16[1][cv] = f[1];
#pragma unroll
      for (int a = 0; a < R8; ++a) sh.qT[a][cv] = f2h(a < R ? q0v[a] : 0.f);          // kernels.py:1573-1577
    }
  }
  if (tid < LPMAX) sh.w[tid] = tid < L ? wv : 0.f;
  __syncthreads();

  // ---- stage 2: B = deq(S0) pn + window, fp16 (kernels.py:1483-1571); the window half by half, as flush_head4.  The fp32
  //      sums keep the order of a whole-window product (hi over every entry, then lo), and the Q rows below that of
  //      16-channel partials: at these ranks one fp16 ulp in B or Q moves 0.1 to 0.3% of a head's codes, and sums in
  //      another order move up to 1.5% over a window or two ----
  f16x4 bh[2][8];                                     // B packed, fp16 (tile layout, k = c for the MFMAs)
  {
    Tile4 t;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int nt = 0; nt < 8; ++nt) t.a[g][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!two) {
      store_half(sh, win, L, 0);
      __syncthreads();
      rebuild_half4x2(t, sh.op[0], sh.op[1], sh.op[2]);
    } else {                                          // hi of both halves, then lo of both: each half staged twice
#pragma unroll 1
      for (int k = 0; k < 4; ++k) {
        if (k) __syncthreads();                       // every wave is past the previous half's operands
        store_half(sh, win, L, k & 1);
        if (k < 3) load_half<KD, VD>(win, st, slot, hv, L, (k + 1) & 1);
        __syncthreads();
        rebuild_half4x1(t, sh.op[0], sh.op[k < 2 ? 1 : 2]);
      }
    }
    load_code_words4<KD, VD>(wds, (const int8_t*)base);
    tile_add_words4(t, wds, sh.svr, sh.skl);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int nt = 0; nt < 8; ++nt) bh[g][nt] = pinned(to_h4(t.a[g][nt]));   // the fp16 rounding of B
  }
  __syncthreads();                                    // every wave is past the rebuild: the operand region is free
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const f16x4 x = colt ? sh.uo16[b][cv] : sh.qo16[b][cv];
#pragma unroll
    for (int i = 0; i < 4; ++i) (colt ? sh.r.uoT : sh.r.qoT)[4 * b + i][cv] = half_bits(x[i]);
  }
  __syncthreads();

  // ---- stage 3: subspace iteration (ITERS = 1) with the algebraic rank-R corrections (kernels.py:1580-1842) ----
  f16x4 bt[2][8];                                     // B^T blocks, formed by the first P step
  {
    const f32x4 p16 = p_step8<true>(sh, bh, bt, pn, R);
#pragma unroll
    for (int i = 0; i < 4; ++i) sh.r.ppT[4 * (q & 1) + i][32 * w + 16 * (q >> 1) + l16] = f2h(p16[i]);
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  // Q = B P16 + pn Q_old (U_old^T P16), columns 4 b .. 4 b + 3 at a time (one MFMA's partial per 16 channels; the waves
  // 2 b, 2 b + 1 then sum the rows, one per thread)
#pragma unroll 1
  for (int b = 0; b < 2; ++b) {
    f16x4 ap[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) ap[g] = *(const f16x4*)&sh.r.ppT[l16 & 7][32 * w + 16 * g + 4 * q];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f32x4 d = mma16(ap[g], bh[g][nt], f32x4{0.f, 0.f, 0.f, 0.f});
        if (q == b) sh.r.qpart[2 * w + g][16 * nt + l16] = d;
      }
    __syncthreads();
    if ((w >> 1) == b) {
      float M2[R8][4];                                // U_old^T P16 over all 128 channels
      gram8(sh, sh.r.uoT, sh.r.ppT, b, M2);
      f32x4 s = sh.r.qpart[0][cv];
#pragma unroll
      for (int k = 1; k < 2 * NW4; ++k) s += sh.r.qpart[k][cv];
      const f32x4 corr = row_times(sh.qo16[0][cv], sh.qo16[1][cv], M2);
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = 4 * b + i < R ? s[i] + pn * corr[i] : 0.f;
      sh.r.qv[b][cv] = s;
    }
    __syncthreads();
  }
  cholqr8_pass(sh, [&](int v, f32x4 y0, f32x4 y1) {
    sh.r.qv[0][v] = y0;
    sh.r.qv[1][v] = y1;
  });
  cholqr8_pass(sh, [&](int v, f32x4 y0, f32x4 y1) {   // fp16 Q; columns past R are zero already
    const f16x4 h0 = to_h4(y0), h1 = to_h4(y1);
    sh.r.qn16[0][v] = h0;
    sh.r.qn16[1][v] = h1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sh.qT[i][v] = half_bits(h0[i]);
      sh.qT[4 + i][v] = half_bits(h1[i]);
    }
  });
  const f32x4 u16 = p_step8<false>(sh, bh, bt, pn, R);   // U16 = P step with Q16
#pragma unroll
  for (int i = 0; i < 4; ++i) sh.r.ppT[4 * (q & 1) + i][32 * w + 16 * (q >> 1) + l16] = f2h(u16[i]);

  // ---- stage 4: residual E = fp16(pn (B / pn + Q_old U_old^T) - Q U^T) (kernels.py:1888-1928), kept packed in B's
  //      registers; the A operands' columns a, r are lanes q < 2, group 1's -U16 from lanes 32 .. 63 ----
  {
    const f16x4 z4 = {};
    const uint2 x = h4_words(to_h4(-u16));
    uint32_t a0 = x.x, b0 = x.x, a1 = x.y, b1 = x.y;
    swap32(a0, b0);                                   // b0, b1 of lanes 0-31: the words of lanes 32-63
    swap32(a1, b1);
    f16x4 auo[2], aun[2];
    aun[0] = q < 2 ? __builtin_bit_cast(f16x4, x) : z4;
    aun[1] = q < 2 ? __builtin_bit_cast(f16x4, make_uint2(b0, b1)) : z4;
#pragma unroll
    for (int g = 0; g < 2; ++g) auo[g] = q < 2 ? sh.uo16[q & 1][32 * w + 16 * g + l16] : z4;
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
      const int v = 16 * nt + l16;
      const f16x4 bqo = sh.qo16[q & 1][v];            // rows a, r >= 8 (lanes q >= 2) meet the zero columns of A
      const f16x4 bqn = sh.r.qn16[q & 1][v];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f16x4 b = bh[g][nt];
        f32x4 e = {h4mul<0>(b, rpn), h4mul<1>(b, rpn), h4mul<2>(b, rpn), h4mul<3>(b, rpn)};
        e = mma16(auo[g], bqo, e);
        e *= pn;
        e = mma16(aun[g], bqn, e);
        bh[g][nt] = to_h4(e);                                                         // E, fp16
      }
    }
  }
  int next = 0;                                       // dynamic schedule: this workgroup's next candidate
  store_codes4<KD, VD>(sh, bh, base, qmax, sched, next);
  // ---- stage 7: factors, window reset (kernels.py:1836-1842, 2014-2025) ----
#pragma unroll
  for (int k = 0; k < 2; ++k) {                       // [U_r | Q_r], row r = tid / 64 + 4 k, 8 bytes per thread
    const int r = (tid >> 6) + 4 * k, c4 = 4 * (tid & 63);
    if (r < R) {
      const uint2 x = c4 < KD ? *(const uint2*)&sh.r.ppT[r][c4] : *(const uint2*)&sh.qT[r][c4 - KD];
      *(uint2*)&UQ[r * (KD + VD) + c4] = x;
    }
  }
  if (tid < L) st.Wbuf[sh_ * L + tid] = 0.f;
  if (tid == 0) {
    st.Pbuf[sh_] = 1.f;
    st.hcnt[sh_] = 0;
    if (sched) sh.due = (unsigned long long)sched_candidate(take_result(next));
  }
  __syncthreads();                                    // LDS reuse by the next head of this workgroup
}

}  // namespace lqf
}  // namespace
