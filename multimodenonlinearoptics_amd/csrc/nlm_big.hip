// nlm_big.hip -- Chi3GNLSE batches whose transforms are staged through HBM/L2,
// and the differentiable (checkpointed forward + adjoint) Chi3GNLSE batch.
//
// Staged transform.  A field of N = P * M points is transformed in two kernels
// (four-step FFT, M in LDS, P in registers):
//
//   X[k1 + P k2] = sum_n2 W_M^(n2 k2) [ W_N^(n2 k1) sum_n1 W_P^(n1 k1) x[n1 M + n2] ]
//
// "mix" kernels (one thread per n2 of a field) apply the radix-P butterflies
// across the P blocks, fused with the pointwise time-domain work that sits between
// two transforms; "conv" kernels (one workgroup per (field, k1)) apply the W_N
// twiddles, run the M-point transform in LDS (nlm_fft.hpp), do the pointwise
// spectral work in the same k1-major order, and transform back.  Between them the
// data sit in the exchange arrays X, Z ([field][k1][n2], coalesced on both sides).
//
// Step (solvers/Chi3GNLSE.cpp:39-92 inside src/_NonlinearMedium.hpp:205-215).  The state and
// the RK4 sum are spectra (A, ACC): a stage is conv (Raman), mix (v y), conv (filter, RK4
// sum, next stage input), mix (|y|^2); the last stage's conv goes on to the dispersion phase,
// so a step is 8 conv + 8 mix launches.  |y|^2 and the Raman convolution v are real where the
// Raman response is the spectrum of a real one (checked when the plan is made; any other
// response takes complex exchanges): blocks k1 and P - k1 are then conjugate, so only
// k1 = 0..P/2 are exchanged and transformed, 0 and P/2 as real numbers.
//
// The launches are bound by the exchange traffic (most of it served by L2 and the Infinity
// Cache) when rows fill the chip (a stage's conv of 64 rows N = 16384 moves 75 MB in 19 us, the
// rate of a large copy), and by the chain of launches, about 4 us each, when they do not.
// Gradient, 19 steps, from 9 conv + 9 mix of one time-domain state with complex exchanges and
// M = 4096 (M = N up to 8192): N = 16384, 64 rows 28.4 -> 12.4 ms; N = 8192, 8 rows 22.9 -> 4.7;
// N = 4096, 40 rows 10.7 -> 4.7; N = 1024, 8 rows 4.9 -> 3.5.
//
// Adjoint.  Gradients use g_z = dL/dRe z + i dL/dIm z.  The forward keeps the
// state's spectrum every K steps.  The reverse sweep takes the segments last
// to first: it recomputes the segment from its checkpoint, storing per step the
// state a, the stage inputs y2, y3, y4 and the Raman convolutions v1..v4, then
// walks the segment backwards.  With f(y) = IFFT(H FFT(y v)), v = IFFT(R FFT(r |y|^2))
// (H = nl0 + nl1 omega, R the Raman response), the adjoint of one stage is
//   g_u = IFFT(conj(H) FFT(g_k)),  g_s = Re IFFT(conj(R) FFT(conj(y) g_u)),
//   g_y = conj(v) g_u + 2 r y g_s,
// and of the dispersion step FFT(g) -> conj(D) FFT(g).  The gradients of the state and of
// the k's are kept as spectra too (GA, GP), again 8 conv + mix pairs per step.
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "nlm_internal.hpp"
#include "nlm_prop.hpp"

namespace {

constexpr int MIX_THREADS = 128;

// mix kinds (mode & 15; mode >> 4 = RK stage 0..3)
enum MixKind {
  MIX_IN = 0,   // X = fwd(input row)
  MIX_RAMAN,    // v = raman conv; X = fwd(v y)
  MIX_STAGE,    // y = stage input st + 1; X = fwd(r |y|^2)
  MIX_STATE,    // state a_i; X = fwd(r0 |a_i|^2) of step i+1
  MIX_ADJ_IN,   // X = fwd(g_out row) (time-domain output)
  MIX_ADJ_U,    // g_u: TMP = conj(v) g_u; X = fwd(conj(y) g_u)
  MIX_ADJ_S,    // g_s: X = fwd(g_y), g_y = TMP + 2 r y Re g_s
  MIX_ADJ_OUT   // g_in = finished transform (time-domain input)
};
// conv operations; those up to CV_FROM_X transform X first
enum ConvOp {
  CV_RAMAN = 0,   // Z = bwd(R fwd X)
  CV_RAMAN_ADJ,   // Z = bwd(conj(R) fwd X)
  CV_STAGE,       // K = H fwd X; RK4 sum and next stage input, after stage 3 the dispersion step
  CV_IN_TIME,     // A = halfIn fwd X
  CV_ADJ_IN_TIME, // fwd X is the gradient of the output
  CV_ADJ_STAGE,   // fwd X is the spectrum of g_y of stage st
  CV_FROM_X = CV_ADJ_STAGE,
  CV_IN_FREQ,     // A = halfIn in
  CV_RESUME,      // A = checkpoint
  CV_ADJ_IN_FREQ, // N g_out is the gradient of the output
  CV_ADJ_RESUME,  // GA is the gradient of a_i
  CV_ADJ_OUT_TIME,  // Z = bwd(conj(halfIn) GA)
  CV_ADJ_OUT_FREQ   // g_in = conj(halfIn) GA / N
};
constexpr int CV_STOP = 4;  // stage argument of CV_ADJ_STAGE: stage 0, the segment's last
enum Table { TAB_RAMAN = 0, TAB_FILTER, TAB_DISP, TAB_IN, TAB_DISP_OUT };

struct BigParams {
  int B, nSteps, N, P, LM;  // N = P 2^LM
  int real;                 // real Raman convolution
  const BigArgs* args;      // of the replayed graph
  cplx* A;                  // [B][P][M] spectrum of the state
  cplx* ACC;                // [B][P][M] spectrum of a + (k1 + 2 k2 + 2 k3) / 6
  cplx* Y;                  // [B][N] stage input y (time, natural order)
  cplx* X;                  // [B][P][M] transform input exchange
  cplx* Z;                  // [B][P][M] transform output exchange
  const cplx* twN;          // W_N^k
  const cplx* twM;          // W_M^k
  const cplx* Hp;           // [5][P][M] frequency responses, k1-major
  const cplx* coef;         // [nZ][3], .re = relative intensity of the stage
  const cplx* in;           // [B][inCols]
  int inCols, inPos;
  cplx* out;                // [B][nOut*N] or nullptr (recomputation); a replay's is in args
  int nOut, outPos, outTime;
  // checkpoints [B][nSeg][P][M] of the spectra of the states a_{sK}
  cplx* ckpt;
  int ckptEvery, nSeg, ckptWrite;
  // segment storage for steps segFirst+1 .. segLast: a (step start), y2, y3, y4 [4][B][N],
  // then v1..v4 [4][B][N] as doubles (real) or complex
  cplx* seg;
  int segFirst, segLast;
  // adjoint work arrays [B][N] and the gradients
  cplx* GP;
  cplx* GA;
  cplx* TMP;
  const cplx* gout;  // [B][nOut*N]
  cplx* gin;         // [B][N]
};

__device__ __forceinline__ int step_of(const BigParams& bp, int di, int fixedStep) {
  return fixedStep >= 0 ? fixedStep : bp.args->step + di;
}
__device__ __forceinline__ cplx* out_of(const BigParams& bp, int fixedStep) {
  return fixedStep >= 0 ? bp.out : bp.args->out;
}

__device__ __forceinline__ bool seg_has(const BigParams& bp, int i) {
  return bp.seg != nullptr && i > bp.segFirst && i <= bp.segLast;
}
template <bool REAL>
__device__ __forceinline__ cplx* seg_step(const BigParams& bp, int i) {
  return bp.seg + (size_t)(i - bp.segFirst - 1) * (REAL ? 6 : 8) * ((size_t)bp.B * bp.N);
}
template <bool REAL>
__device__ __forceinline__ cplx* seg_y(const BigParams& bp, int i, int st) {
  return seg_step<REAL>(bp, i) + st * ((size_t)bp.B * bp.N);
}
template <bool REAL>
__device__ __forceinline__ void seg_put_v(const BigParams& bp, int i, int st, size_t q, cplx v) {
  const size_t BN = (size_t)bp.B * bp.N;
  cplx* base = seg_step<REAL>(bp, i) + 4 * BN;
  if constexpr (REAL) __builtin_nontemporal_store(v.re, (double*)base + st * BN + q);
  else store_stream(base + st * BN + q, v);
}
template <bool REAL>
__device__ __forceinline__ cplx seg_get_v(const BigParams& bp, int i, int st, size_t q) {
  const size_t BN = (size_t)bp.B * bp.N;
  const cplx* base = seg_step<REAL>(bp, i) + 4 * BN;
  if constexpr (REAL) return mk(__builtin_nontemporal_load((const double*)base + st * BN + q), 0.0);
  else return load_stream(base + st * BN + q);
}

// relative intensity of RK stage st of step i (prev, intermediate x2, current)
__device__ __forceinline__ double stage_r(const BigParams& bp, int i, int st) {
  return bp.coef[(size_t)i * 3 + (st == 0 ? 0 : st == 3 ? 2 : 1)].re;
}

// DFT across the P blocks, in natural order.
template <int P, bool INV>
__device__ __forceinline__ void dft_blocks(cplx (&v)[P]) {
  if constexpr (P == 16) {  // 4 x 4: n = 4 a + b, k = c + 4 d
    constexpr double C1 = 0.92387953251128675613, S1 = 0.38268343236508977173, R = 0.70710678118654752440;
    constexpr cplx W[10] = {{1, 0}, {C1, -S1}, {R, -R}, {S1, -C1}, {0, -1}, {-S1, -C1}, {-R, -R}, {-C1, -S1}, {-1, 0}, {-C1, S1}};
    cplx u[16];
#pragma unroll
    for (int b = 0; b < 4; b++) {
#pragma unroll
      for (int a = 0; a < 4; a++) u[4 * b + a] = v[4 * a + b];
      dft_small<4, INV>(u + 4 * b);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
      cplx x[4];
#pragma unroll
      for (int b = 0; b < 4; b++) x[b] = b * c == 0 ? u[4 * b + c] : twmul<INV>(u[4 * b + c], W[b * c]);
      dft_small<4, INV>(x);
#pragma unroll
      for (int d = 0; d < 4; d++) v[c + 4 * d] = x[d];
    }
  } else if constexpr (P > 1) {
    dft_small<P, INV>(v);
  }
}

// Exchange of one n2 across the blocks: all of them as complex numbers, or (REAL) the
// independent half of a real sequence, blocks 0 and P/2 as doubles.
template <int P, bool REAL>
__device__ __forceinline__ void get_blocks(cplx (&v)[P], const cplx* Z, size_t fo, int M, int n2) {
  if constexpr (REAL) {
    v[0] = mk(reinterpret_cast<const double*>(Z + fo)[n2], 0.0);
    if constexpr (P > 1) v[P / 2] = mk(reinterpret_cast<const double*>(Z + fo + (size_t)(P / 2) * M)[n2], 0.0);
#pragma unroll
    for (int k = 1; k < (P + 1) / 2; k++) {
      v[k] = Z[fo + (size_t)k * M + n2];
      v[P - k] = conj(v[k]);
    }
  } else {
#pragma unroll
    for (int k = 0; k < P; k++) v[k] = Z[fo + (size_t)k * M + n2];
  }
}
template <int P, bool REAL>
__device__ __forceinline__ void put_blocks(const cplx (&v)[P], cplx* X, size_t fo, int M, int n2) {
  if constexpr (REAL) {
    reinterpret_cast<double*>(X + fo)[n2] = v[0].re;
    if constexpr (P > 1) reinterpret_cast<double*>(X + fo + (size_t)(P / 2) * M)[n2] = v[P / 2].re;
#pragma unroll
    for (int k = 1; k < (P + 1) / 2; k++) X[fo + (size_t)k * M + n2] = v[k];
  } else {
#pragma unroll
    for (int k = 0; k < P; k++) X[fo + (size_t)k * M + n2] = v[k];
  }
}

// The field and the part of it that a workgroup works on.  Workgroups go to the eight XCDs in
// turn, so eight fields at a time are interleaved: a field's parts, in every launch, fall
// on the same XCD and find the field's exchange arrays in its L2 (batch N = 8192, 64 rows
// 172 -> 148 us per step; gradient N = 4096, 40 rows 292 -> 256, N = 16384, 64 rows 688 -> 659).
struct Place {
  int f, part;
};
__device__ __forceinline__ Place place(int fields, int parts) {
  const int b = blockIdx.x, g = b / (8 * parts), r = b - g * 8 * parts;
  const int n = min(8, fields - 8 * g);
  return {8 * g + r % n, r / n};
}

template <int P, bool REAL>
__global__ void __launch_bounds__(MIX_THREADS) k_big_mix(BigParams bp, int mode, int di, int fixedStep) {
  const int i = step_of(bp, di, fixedStep);
  if (fixedStep < 0 && i > bp.nSteps) return;
  const int M = 1 << bp.LM, N = bp.N;
  int f, n2;
  if (M >= MIX_THREADS) {
    const Place p = place(bp.B, M / MIX_THREADS);
    f = p.f;
    n2 = p.part * MIX_THREADS + threadIdx.x;
  } else {
    const long gid = (long)blockIdx.x * MIX_THREADS + threadIdx.x;
    if (gid >= ((long)bp.B << bp.LM)) return;
    f = (int)(gid >> bp.LM);
    n2 = (int)(gid & (M - 1));
  }
  const size_t fo = (size_t)f * N;
  const int kind = mode & 15, st = mode >> 4;
  const double s = 1.0 / N;
  // the operands of the pointwise work are loaded together with the blocks
  cplx v[P], e[P], g[P];
  if (kind == MIX_IN || kind == MIX_ADJ_IN) {
    const cplx* src = kind == MIX_IN ? bp.in + (size_t)f * bp.inCols + (size_t)bp.inPos * N
                                     : bp.gout + (size_t)f * bp.nOut * N + (size_t)bp.outPos * N;
#pragma unroll
    for (int n1 = 0; n1 < P; n1++) v[n1] = src[n1 * M + n2];
  } else {
    if (kind == MIX_RAMAN || kind == MIX_ADJ_S) get_blocks<P, REAL>(v, bp.Z, fo, M, n2);
    else get_blocks<P, false>(v, bp.Z, fo, M, n2);
    if (kind == MIX_RAMAN) {
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) e[n1] = bp.Y[fo + n1 * M + n2];
    } else if (kind == MIX_ADJ_U) {
      const cplx* ys = seg_y<REAL>(bp, i, st);
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) {
        const size_t q = fo + n1 * M + n2;
        g[n1] = seg_get_v<REAL>(bp, i, st, q);  // last read of v_s
        e[n1] = ys[q];                          // y_s is read again by MIX_ADJ_S
      }
    } else if (kind == MIX_ADJ_S) {
      const cplx* ys = seg_y<REAL>(bp, i, st);
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) {
        const size_t q = fo + n1 * M + n2;
        g[n1] = bp.TMP[q];
        e[n1] = load_stream(ys + q);  // last read of y_s
      }
    }
    dft_blocks<P, true>(v);
#pragma unroll
    for (int n1 = 0; n1 < P; n1++) v[n1] = v[n1] * s;
  }
  bool real = false;  // what goes into X is real
  switch (kind) {
    case MIX_RAMAN: {
      const bool keep = seg_has(bp, i);
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) {
        const size_t q = fo + n1 * M + n2;
        if (keep) seg_put_v<REAL>(bp, i, st, q, v[n1]);
        v[n1] = REAL ? v[n1].re * e[n1] : v[n1] * e[n1];
      }
      break;
    }
    case MIX_STAGE:
    case MIX_STATE: {
      const bool state = kind == MIX_STATE;
      if (state && i == bp.nSteps) {
        cplx* out = out_of(bp, fixedStep);
        if (out && bp.outTime) {
#pragma unroll
          for (int n1 = 0; n1 < P; n1++)
            out[(size_t)f * bp.nOut * N + (size_t)bp.outPos * N + n1 * M + n2] = v[n1];
        }
        return;
      }
      const int step = state ? i + 1 : i, next = state ? 0 : st + 1;
      const double r = stage_r(bp, step, next);
      const bool keep = seg_has(bp, step);
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) {
        const size_t q = fo + n1 * M + n2;
        bp.Y[q] = v[n1];
        if (keep) store_stream(seg_y<REAL>(bp, step, next) + q, v[n1]);
        v[n1] = mk(r * abs2(v[n1]), 0.0);
      }
      real = true;
      break;
    }
    case MIX_ADJ_U:
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) {
        bp.TMP[fo + n1 * M + n2] = REAL ? g[n1].re * v[n1] : conj(g[n1]) * v[n1];
        v[n1] = conj(e[n1]) * v[n1];
        if (REAL) v[n1].im = 0.0;  // only the real part of the convolution is used
      }
      real = true;
      break;
    case MIX_ADJ_S: {
      const double r2 = 2.0 * stage_r(bp, i, st);
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) v[n1] = g[n1] + (r2 * v[n1].re) * e[n1];
      break;
    }
    case MIX_ADJ_OUT:
#pragma unroll
      for (int n1 = 0; n1 < P; n1++) bp.gin[fo + n1 * M + n2] = v[n1];
      return;
    default:  // MIX_IN, MIX_ADJ_IN
      break;
  }
  dft_blocks<P, false>(v);
  if (REAL && real) put_blocks<P, REAL>(v, bp.X, fo, M, n2);
  else put_blocks<P, false>(v, bp.X, fo, M, n2);
}

// One block of M points.  The operations come in four kernels, so that each holds only the
// registers it needs (256 per lane, two waves per SIMD): the rows of the spectral work are
// fetched before the last exchange of the forward transform, the W_N twiddles once per side.
enum ConvClass { CLS_RAMAN, CLS_STAGE, CLS_ADJ, CLS_ENDS };
constexpr ConvClass conv_class(int op) {
  return op <= CV_RAMAN_ADJ ? CLS_RAMAN : op == CV_STAGE ? CLS_STAGE : op == CV_ADJ_STAGE ? CLS_ADJ : CLS_ENDS;
}

template <int LM, int CLS>
__global__ void __launch_bounds__((FftShape<LM>::T), (2)) k_big_conv(BigParams bp, int op, int st, int di, int fixedStep) {
  using F = FftShape<LM>;
  constexpr int T = F::T, M = F::N;
  __shared__ cplx lds[F::lds_elems];
  const int i = step_of(bp, di, fixedStep);
  if (fixedStep < 0 && i > bp.nSteps) return;
  const int P = bp.P, N = bp.N;
  const unsigned t = threadIdx.x;
  const bool half = CLS == CLS_RAMAN && bp.real;
  const int blocks = half ? P / 2 + 1 : P;
  const Place p = place(bp.B, blocks);
  const int f = p.f, k1 = p.part;
  const bool reals = half && (k1 == 0 || 2 * k1 == P);
  const size_t xo = (size_t)f * N + (size_t)k1 * M;
  const bool last = i == bp.nSteps;
  const auto table = [&](int k) __attribute__((always_inline)) { return bp.Hp + (size_t)k * N + (size_t)k1 * M; };
  const auto load = [&](cplx (&x)[8], const cplx* src) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < 8; m++) x[m] = src[t + T * m];
  };
  const auto load_w = [&](cplx (&w)[8]) __attribute__((always_inline)) {  // W_N^(n2 k1)
#pragma unroll
    for (int m = 0; m < 8; m++) w[m] = bp.twN[(t + T * m) * k1];
  };
  cplx v[8];
  const auto put = [&](cplx* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < 8; m++) (dst + xo)[t + T * m] = v[m];
  };
  // natural-order rows of the caller, element k1 + P k2
  const auto at = [&](int m) __attribute__((always_inline)) { return (size_t)k1 + (size_t)P * (t + T * m); };
  const size_t ckptRow = (((size_t)f * bp.nSeg + i / bp.ckptEvery) * N) + (size_t)k1 * M;

  const bool fromX = op <= CV_FROM_X;
  cplx w[8];
  if (fromX) {
    if (reals) {
      const double* x = reinterpret_cast<const double*>(bp.X + xo);
#pragma unroll
      for (int m = 0; m < 8; m++) v[m] = mk(x[t + T * m], 0.0);
    } else {
      load(v, bp.X + xo);
    }
    if (k1) load_w(w);
  }
  RegTwiddles<LM> tw;
  fft_load_twiddles<LM>(tw.w, bp.twM, t);
  if (fromX && k1) {
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = v[m] * w[m];
  }

  // v becomes the spectral input of the inverse transform; begin: v is the gradient of the
  // state after step i, the adjoint of that step starts
  bool begin = false;
  int beginTable = TAB_DISP;
  if constexpr (CLS == CLS_RAMAN) {
    cplx h[8];
    fft_field1<LM, false, (T <= 64)>(v, lds, t, tw,
                                     [&]() __attribute__((always_inline)) { load(h, table(TAB_RAMAN)); });
    const double sign = op == CV_RAMAN ? 1.0 : -1.0;
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = v[m] * mk(h[m].re, sign * h[m].im);
  } else if constexpr (CLS == CLS_STAGE) {
    cplx h[8], a[8], c[8];
    fft_field1<LM, false, (T <= 64)>(v, lds, t, tw, [&]() __attribute__((always_inline)) {
      load(h, table(TAB_FILTER));
      if (st < 3) load(a, bp.A + xo);
      if (st > 0) load(c, bp.ACC + xo);
    });
    if (st < 3) {
      const double wy = st == 2 ? 1.0 : 0.5;
#pragma unroll
      for (int m = 0; m < 8; m++) {
        const cplx k = v[m] * h[m];
        (bp.ACC + xo)[t + T * m] = st == 0 ? a[m] + k * (1. / 6.) : c[m] + k * (1. / 3.);
        v[m] = a[m] + wy * k;
      }
    } else {
      const cplx* D = table(last ? TAB_DISP_OUT : TAB_DISP);  // the last step goes half a step out
#pragma unroll
      for (int m = 0; m < 8; m++) v[m] = (c[m] + (v[m] * h[m]) * (1. / 6.)) * D[t + T * m];
      if (last && !bp.outTime) {
        if (cplx* out = out_of(bp, fixedStep)) {
#pragma unroll
          for (int m = 0; m < 8; m++) out[(size_t)f * bp.nOut * N + (size_t)bp.outPos * N + at(m)] = v[m];
        }
        return;
      }
      if (!last) put(bp.A);
      if (bp.ckptWrite && !last && i % bp.ckptEvery == 0) {
#pragma unroll
        for (int m = 0; m < 8; m++) store_stream(bp.ckpt + ckptRow + t + T * m, v[m]);
      }
    }
  } else if constexpr (CLS == CLS_ADJ) {
    const bool start = st == 0 || st == CV_STOP;
    cplx h[8], a[8], c[8];
    fft_field1<LM, false, (T <= 64)>(v, lds, t, tw, [&]() __attribute__((always_inline)) {
      if (st != 3) load(a, bp.GA + xo);
      if (!start) {
        load(h, table(TAB_FILTER));
        load(c, bp.GP + xo);
      }
    });
    if (start) {
#pragma unroll
      for (int m = 0; m < 8; m++) v[m] = a[m] + v[m];
      if (st == CV_STOP) {
        put(bp.GA);
        return;
      }
      begin = true;
    } else {
      // k3 feeds y4 = a + k3, k2 feeds y3 = a + k2/2, k1 feeds y2 = a + k1/2
      const double wp = st == 1 ? 1. / 6. : 1. / 3., wy = st == 3 ? 1.0 : 0.5;
#pragma unroll
      for (int m = 0; m < 8; m++) {
        (bp.GA + xo)[t + T * m] = (st == 3 ? c[m] : a[m]) + v[m];  // GP is the first term
        v[m] = (c[m] * wp + v[m] * wy) * conj(h[m]);
      }
    }
  } else {
    if (fromX) fft_field1<LM, false, (T <= 64)>(v, lds, t, tw);
    if (op == CV_IN_TIME || op == CV_IN_FREQ || op == CV_RESUME) {
      if (op == CV_RESUME) {
        load(v, bp.ckpt + ckptRow);
      } else {
        if (op == CV_IN_FREQ) {
#pragma unroll
          for (int m = 0; m < 8; m++) v[m] = bp.in[(size_t)f * bp.inCols + (size_t)bp.inPos * N + at(m)];
        }
        const cplx* H = table(TAB_IN);
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = v[m] * H[t + T * m];
        if (bp.ckptWrite) {
#pragma unroll
          for (int m = 0; m < 8; m++) store_stream(bp.ckpt + ckptRow + t + T * m, v[m]);
        }
      }
      put(bp.A);
    } else if (op == CV_ADJ_OUT_TIME || op == CV_ADJ_OUT_FREQ) {
      load(v, bp.GA + xo);
      const cplx* H = table(TAB_IN);
      const double s = op == CV_ADJ_OUT_FREQ ? 1.0 / N : 1.0;
#pragma unroll
      for (int m = 0; m < 8; m++) v[m] = (v[m] * conj(H[t + T * m])) * s;
      if (op == CV_ADJ_OUT_FREQ) {
#pragma unroll
        for (int m = 0; m < 8; m++) bp.gin[(size_t)f * N + at(m)] = v[m];
        return;
      }
    } else {
      begin = true;
      if (op == CV_ADJ_RESUME) {
        load(v, bp.GA + xo);
      } else {
        beginTable = TAB_DISP_OUT;
        if (op == CV_ADJ_IN_FREQ) {
#pragma unroll
          for (int m = 0; m < 8; m++)
            v[m] = bp.gout[(size_t)f * bp.nOut * N + (size_t)bp.outPos * N + at(m)] * (double)N;
        }
      }
    }
  }
  if ((CLS == CLS_ADJ || CLS == CLS_ENDS) && begin) {
    const cplx *D = table(beginTable), *Hf = table(TAB_FILTER);
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = v[m] * conj(D[t + T * m]);
    put(bp.GP);
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = (v[m] * (1. / 6.)) * conj(Hf[t + T * m]);
  }
  // from M = 512 the lane's twiddles are read again, so that they are not live across the
  // spectral work (with them it spilled)
  if constexpr (LM >= 9 && CLS != CLS_RAMAN) fft_load_twiddles<LM>(tw.w, bp.twM, opaque_lane((int)t));
  fft_field1<LM, true, (T <= 64)>(v, lds, t, tw, [&]() __attribute__((always_inline)) {
    if (k1) load_w(w);
  });  // unscaled; the mix kernel applies 1/N
  if (k1) {
#pragma unroll
    for (int m = 0; m < 8; m++) v[m] = v[m] * conj(w[m]);
  }
  if (reals) {
    double* z = reinterpret_cast<double*>(bp.Z + xo);
#pragma unroll
    for (int m = 0; m < 8; m++) z[t + T * m] = v[m].re;
  } else {
    put(bp.Z);
  }
}

__global__ void k_big_set_args(BigArgs* a, BigArgs value) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *a = value;
}
__global__ void k_big_advance(BigArgs* a, int steps) {
  if (blockIdx.x == 0 && threadIdx.x == 0) a->step += steps;
}

// Hp[tab][k1 M + k2] = H[k1 + P k2]  (tab 4: disp * halfOut)
__global__ void k_big_perm(const cplx* __restrict__ ram, const cplx* __restrict__ flt, const cplx* __restrict__ ds,
                           const cplx* __restrict__ hin, const cplx* __restrict__ hout, int N, int P, int M,
                           cplx* __restrict__ Hp) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  const int k1 = j / M, k2 = j % M, k = k1 + P * k2;
  Hp[j] = ram[k];
  Hp[(size_t)N + j] = flt[k];
  Hp[2 * (size_t)N + j] = ds[k];
  Hp[3 * (size_t)N + j] = hin[k];
  Hp[4 * (size_t)N + j] = ds[k] * hout[k];
}

// Launch shape: N = P 2^LM and the kernels of that split.
struct Stager {
  int P = 0, LM = 0;
  void (*mix)(const BigParams&, int, int, int, hipStream_t) = nullptr;
  void (*conv)(const BigParams&, int, int, int, int, hipStream_t) = nullptr;
};

template <int P>
void launch_mix(const BigParams& bp, int mode, int di, int fixed, hipStream_t s) {
  const dim3 g((unsigned)((((long)bp.B << bp.LM) + MIX_THREADS - 1) / MIX_THREADS));
  if (bp.real) hipLaunchKernelGGL((k_big_mix<P, true>), g, dim3(MIX_THREADS), 0, s, bp, mode, di, fixed);
  else hipLaunchKernelGGL((k_big_mix<P, false>), g, dim3(MIX_THREADS), 0, s, bp, mode, di, fixed);
}
template <int LM>
void launch_conv(const BigParams& bp, int op, int st, int di, int fixed, hipStream_t s) {
  const ConvClass cls = conv_class(op);
  const int blocks = cls == CLS_RAMAN && bp.real ? bp.P / 2 + 1 : bp.P;
  const dim3 g((unsigned)(bp.B * blocks)), b(FftShape<LM>::T);
  if (cls == CLS_RAMAN) hipLaunchKernelGGL((k_big_conv<LM, CLS_RAMAN>), g, b, 0, s, bp, op, st, di, fixed);
  else if (cls == CLS_STAGE) hipLaunchKernelGGL((k_big_conv<LM, CLS_STAGE>), g, b, 0, s, bp, op, st, di, fixed);
  else if (cls == CLS_ADJ) hipLaunchKernelGGL((k_big_conv<LM, CLS_ADJ>), g, b, 0, s, bp, op, st, di, fixed);
  else hipLaunchKernelGGL((k_big_conv<LM, CLS_ENDS>), g, b, 0, s, bp, op, st, di, fixed);
}

// log2 M of the split.  Small blocks fill the chip with few rows and overlap several
// workgroups per CU, large ones need fewer blocks across a mix thread.  Gradient of 19 steps,
// ms:
//   N = 16384, 64 rows: M = 4096 13.8, 2048 12.6, 1024 12.7; 4 rows 8.6, 6.2, 5.9
//   N = 8192, 48 rows: 4096 9.6, 2048 7.2, 1024 7.1, 512 7.1; 8 rows 8.4, 5.9, 5.1, 5.3
//   N = 4096, 48 rows: 2048 5.7, 1024 5.0, 512 4.9, 256 5.7
//   N = 2048 and 1024, 48 rows: 1024 4.4, 4.0; 512 4.0, 3.6; 256 4.5, 4.1
int split_of(int L) { return L <= 12 ? std::min(L, 9) : L <= 14 ? 10 : L - 4; }

Stager pick_stager(int L) {
  Stager st;
  if (L < 5 || L > 15) return st;
  st.LM = split_of(L);
  st.P = 1 << (L - st.LM);
  switch (st.P) {
    case 1: st.mix = &launch_mix<1>; break;
    case 2: st.mix = &launch_mix<2>; break;
    case 4: st.mix = &launch_mix<4>; break;
    case 8: st.mix = &launch_mix<8>; break;
    case 16: st.mix = &launch_mix<16>; break;
  }
  switch (st.LM) {
    case 5: st.conv = &launch_conv<5>; break;
    case 6: st.conv = &launch_conv<6>; break;
    case 7: st.conv = &launch_conv<7>; break;
    case 8: st.conv = &launch_conv<8>; break;
    case 9: st.conv = &launch_conv<9>; break;
    case 10: st.conv = &launch_conv<10>; break;
    case 11: st.conv = &launch_conv<11>; break;
  }
  return st;
}

// One forward step: di = index within a replayed graph (fixed < 0) or the step itself.
// untilV: only as far as the last Raman convolution (the recomputed stage data are complete).
void launch_step(const Stager& sg, const BigParams& bp, int di, int fixed, hipStream_t s, bool untilV = false) {
  for (int st = 0; st < 4; st++) {
    sg.conv(bp, CV_RAMAN, st, di, fixed, s);
    sg.mix(bp, MIX_RAMAN | (st << 4), di, fixed, s);
    if (untilV && st == 3) return;
    sg.conv(bp, CV_STAGE, st, di, fixed, s);
    sg.mix(bp, st < 3 ? MIX_STAGE | (st << 4) : MIX_STATE, di, fixed, s);
  }
}

void launch_prologue(const Stager& sg, const BigParams& bp, bool inTime, hipStream_t s) {
  if (inTime) {
    sg.mix(bp, MIX_IN, 0, 0, s);
    sg.conv(bp, CV_IN_TIME, 0, 0, 0, s);
  } else {
    sg.conv(bp, CV_IN_FREQ, 0, 0, 0, s);
  }
  sg.mix(bp, MIX_STATE, 0, 0, s);
}

// The adjoint of forward steps i1 .. i0 + 1; GA holds the gradient of a_{i1}'s spectrum unless
// i1 is the last step, and that of a_{i0}'s afterwards.
void launch_adjoint_segment(const Stager& sg, const BigParams& bp, int i0, int i1, hipStream_t s) {
  if (i1 < bp.nSteps) {
    sg.conv(bp, CV_ADJ_RESUME, 0, 0, i1, s);
  } else if (bp.outTime) {
    sg.mix(bp, MIX_ADJ_IN, 0, i1, s);
    sg.conv(bp, CV_ADJ_IN_TIME, 0, 0, i1, s);
  } else {
    sg.conv(bp, CV_ADJ_IN_FREQ, 0, 0, i1, s);
  }
  for (int i = i1; i > i0; i--)
    for (int st = 3; st >= 0; st--) {
      sg.mix(bp, MIX_ADJ_U | (st << 4), 0, i, s);
      sg.conv(bp, CV_RAMAN_ADJ, st, 0, i, s);
      sg.mix(bp, MIX_ADJ_S | (st << 4), 0, i, s);
      sg.conv(bp, CV_ADJ_STAGE, st == 0 && i == i0 + 1 ? CV_STOP : st, 0, i, s);
    }
}

int ensure_state(nlm_plan* p, int rows) {
  int e;
  if ((e = p->bigState.ensure(5 * (size_t)rows * p->N)) || (e = p->bigH.ensure(5 * (size_t)p->N))) return e;
  return p->bigArgs.ensure(1);
}

int setup_params(nlm_plan* p, const Stager& sg, int rows, BigParams& bp) {
  const int N = p->N;
  const size_t BN = (size_t)rows * N;
  int e;
  if ((e = scratch_wait(p)) || (e = ensure_state(p, rows))) return e;
  const cplx* twM = nullptr;
  if ((e = get_twiddles(1 << sg.LM, &twM))) return e;
  hipLaunchKernelGGL(k_big_perm, dim3((N + 255) / 256), dim3(256), 0, p->stream, p->raman.p, p->filt.p, p->dstep.p,
                     p->halfIn.p, p->halfOut.p, N, sg.P, 1 << sg.LM, p->bigH.p);
  HIP_TRY(hipGetLastError());
  std::memset(&bp, 0, sizeof bp);
  bp.B = rows;
  bp.nSteps = p->nZ - 1;
  bp.N = N;
  bp.P = sg.P;
  bp.LM = sg.LM;
  bp.real = p->ramanReal;
  bp.args = p->bigArgs.p;
  bp.A = p->bigState.p;
  bp.Y = bp.A + BN;
  bp.ACC = bp.Y + BN;
  bp.X = bp.ACC + BN;
  bp.Z = bp.X + BN;
  bp.twN = p->tw;
  bp.twM = twM;
  bp.Hp = p->bigH.p;
  bp.coef = p->coef.p;
  bp.ckptEvery = 1;
  bp.nSeg = 1;
  return NLM_OK;
}

}  // namespace

// Steps per captured graph.
static constexpr int BIG_GRAPH_STEPS = 32;  // at most, see below

bool nlm_big_supported(int model, int L) { return model == NLM_CHI3GNLSE && (L == 14 || L == 15); }

// N = 8192 also fits one workgroup's LDS, with 1024 lanes of 128 registers that spill and one
// CU per row: 4 rows 307 us per step against 72 staged, 64 rows 385 against 148, 128 rows 424
// against 246, 256 rows about 430 against 391.  With more rows than CUs the two are close, and
// the in-LDS kernel needs no state arrays in memory; it also runs when these do not fit, and
// under a caller's stream capture, where it is one plain launch.  At N = 4096 it is the faster
// one (4 rows 55 against 61, 64 rows 70 against 95).
bool nlm_big_better(nlm_plan* p, int rows) {
  if (p->model != NLM_CHI3GNLSE || p->L != 13 || p->nZ < 2 || rows > device_cus()) return false;
  if (stream_capturing(p->stream)) return false;
  if (ensure_state(p, rows) == NLM_OK) return true;
  (void)hipGetLastError();
  return false;
}

// Batch propagation of a Chi3GNLSE plan with nFreqs 8192 (nlm_big_better), 16384 or 32768.
// in / out are device arrays with the layout of nlm_batch_dev.
int nlm_big_batch(nlm_plan* p, const cplx* in, int rows, int cols, int inTime, int inPos, int nOut, int outPos,
                  cplx* out) {
  const Stager sg = pick_stager(p->L);
  if (p->model != NLM_CHI3GNLSE || !sg.mix)
    return set_err(NLM_INVALID_ARGUMENT, "unsupported size for the staged transform");
  if (p->nZ < 2) return set_err(NLM_INVALID_ARGUMENT, "the staged transform needs at least two z steps");
  if (rows == 0) return NLM_OK;
  BigParams bp;
  if (int e = setup_params(p, sg, rows, bp)) return e;
  bp.in = in;
  bp.inCols = cols;
  bp.inPos = inPos;
  bp.out = out;
  bp.nOut = nOut;
  bp.outPos = outPos;
  bp.outTime = inTime;
  launch_prologue(sg, bp, inTime != 0, p->stream);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_big_set_args, dim3(1), dim3(64), 0, p->stream, p->bigArgs.p, BigArgs{1, out});
  HIP_TRY(hipGetLastError());

  // the z loop: a graph of BIG_GRAPH_STEPS steps, rebuilt when the batch's shape or domain
  // changes.  The caller's output buffer is an argument in device memory, not of the graph:
  // 64 rows N = 8192, 32 steps into another buffer than the call before, 5.1 ms with the graph
  // rebuilt (up to 8.4), 4.0 so.  NLM_NO_GRAPH=1 in the environment launches the same kernels
  // directly (for tools that do not follow graph launches)
  const int launches = (p->nZ - 1 + BIG_GRAPH_STEPS - 1) / BIG_GRAPH_STEPS;
  const int G = (p->nZ - 1 + launches - 1) / launches;  // fewest idle steps in the last replay
  const char* noGraph = std::getenv("NLM_NO_GRAPH");
  if (noGraph && noGraph[0] == '1') {
    for (int r = 0; r < launches; r++) {
      for (int di = 0; di < G; di++) launch_step(sg, bp, di, -1, p->stream);
      hipLaunchKernelGGL(k_big_advance, dim3(1), dim3(64), 0, p->stream, p->bigArgs.p, G);
    }
    HIP_TRY(hipGetLastError());
    return NLM_OK;
  }
  if (!p->bigExec || p->bigKey[0] != rows || p->bigKey[1] != cols || p->bigKey[2] != inTime ||
      p->bigKey[3] != inPos || p->bigKey[4] != nOut || p->bigKey[5] != outPos || p->bigStatePtr != p->bigState.p) {
    if (p->bigExec) {
      // an asynchronous call before this one may still be replaying it
      if (!stream_capturing(p->stream)) HIP_TRY(hipStreamSynchronize(p->stream));
      (void)hipGraphExecDestroy(p->bigExec);
    }
    p->bigExec = nullptr;
    hipGraph_t g = nullptr;
    HIP_TRY(hipStreamBeginCapture(p->stream, hipStreamCaptureModeThreadLocal));
    for (int di = 0; di < G; di++) launch_step(sg, bp, di, -1, p->stream);
    hipLaunchKernelGGL(k_big_advance, dim3(1), dim3(64), 0, p->stream, p->bigArgs.p, G);
    const hipError_t ce = hipGetLastError();
    const hipError_t ee = hipStreamEndCapture(p->stream, &g);
    if (ce != hipSuccess || ee != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return set_err(NLM_DEVICE_ERROR,
                     std::string("graph capture failed: ") + hipGetErrorString(ce != hipSuccess ? ce : ee));
    }
    const hipError_t ie = hipGraphInstantiate(&p->bigExec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ie != hipSuccess) {
      p->bigExec = nullptr;
      return set_err(NLM_DEVICE_ERROR, std::string("graph instantiation failed: ") + hipGetErrorString(ie));
    }
    const int key[6] = {rows, cols, inTime, inPos, nOut, outPos};
    std::memcpy(p->bigKey, key, sizeof key);
    p->bigStatePtr = p->bigState.p;
  }
  for (int r = 0; r < launches; r++) HIP_TRY(hipGraphLaunch(p->bigExec, p->stream));
  return NLM_OK;
}

// ---------------------------------------------------------------------------
// differentiable Chi3GNLSE batch (C-ABI)
// ---------------------------------------------------------------------------

static int gnlse_diff_check(nlm_plan* p) {
  if (!p) return set_err(NLM_INVALID_ARGUMENT, "null argument");
  if (p->model != NLM_CHI3GNLSE)
    return set_err(NLM_INVALID_ARGUMENT, "the differentiable batch is implemented for Chi3GNLSE");
  if (!pick_stager(p->L).mix) return set_err(NLM_INVALID_ARGUMENT, "the differentiable batch needs nFreqs a power of two, 32..32768");
  if (p->nZ < 2) return set_err(NLM_INVALID_ARGUMENT, "the differentiable batch needs at least two z steps");
  return NLM_OK;
}

// a result into the caller's host memory, or into its device memory (dev)
static int from_device(nlm_plan* p, double* dst, const cplx* src, size_t bytes, bool dev) {
  if (!dev) {
    const HostCopy c = {dst, src, bytes};
    return nlm_to_host(&c, 1, p->stream);
  }
  HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, p->stream));
  HIP_TRY(hipStreamSynchronize(p->stream));
  return NLM_OK;
}

static int batch_forward(nlm_plan* p, const double* inputs, int rows, int in_time, int ckpt_every, double* out,
                         bool dev);

extern "C" int nlm_batch_forward(nlm_plan* p, const double* inputs, int rows, int in_time, int ckpt_every,
                                 double* out) {
  return batch_forward(p, inputs, rows, in_time, ckpt_every, out, false);
}

static int check_device(nlm_plan* p, const void* a, const void* b) {
  if (!p) return set_err(NLM_INVALID_ARGUMENT, "null plan");
  if (!nlm_on_device(a, p->device) || !nlm_on_device(b, p->device))
    return set_err(NLM_INVALID_ARGUMENT, "not memory of the plan's device");
  return NLM_OK;
}

extern "C" int nlm_batch_forward_dev(nlm_plan* p, const double* inputs_dev, int rows, int in_time, int ckpt_every,
                                     double* out_dev) {
  if (int e = check_device(p, inputs_dev, out_dev)) return e;
  return batch_forward(p, inputs_dev, rows, in_time, ckpt_every, out_dev, true);
}

static int batch_forward(nlm_plan* p, const double* inputs, int rows, int in_time, int ckpt_every, double* out,
                         bool dev) {
  if (int e = gnlse_diff_check(p)) return e;
  if (!inputs || !out || rows <= 0) return set_err(NLM_INVALID_ARGUMENT, "null argument or empty batch");
  const int N = p->N, nSteps = p->nZ - 1;
  int K = ckpt_every;
  if (K <= 0) K = (int)std::ceil(std::sqrt(nSteps / 8.0));
  if (K < 1) K = 1;
  if (K > nSteps) K = nSteps;
  const int nSeg = (nSteps + K - 1) / K;
  const size_t BN = (size_t)rows * N;
  const Stager sg = pick_stager(p->L);
  int e;
  if ((e = p->in.ensure(BN)) || (e = p->out.ensure(BN)) || (e = p->ckpt.ensure((size_t)nSeg * BN))) return e;
  if (dev) HIP_TRY(hipMemcpyAsync(p->in.p, inputs, BN * sizeof(cplx), hipMemcpyDeviceToDevice, p->stream));
  else if ((e = nlm_to_device(p->in.p, inputs, BN * sizeof(cplx), p->stream))) return e;
  BigParams bp;
  if ((e = setup_params(p, sg, rows, bp))) return e;
  bp.in = p->in.p;
  bp.inCols = N;
  bp.inPos = 0;
  bp.out = p->out.p;
  bp.nOut = 1;
  bp.outPos = 0;
  bp.outTime = in_time;
  bp.ckpt = p->ckpt.p;
  bp.ckptEvery = K;
  bp.nSeg = nSeg;
  bp.ckptWrite = 1;
  tic(p, 2);
  launch_prologue(sg, bp, in_time != 0, p->stream);
  for (int i = 1; i <= nSteps; i++) launch_step(sg, bp, 0, i, p->stream);
  HIP_TRY(hipGetLastError());
  tic(p, 3);
  if ((e = from_device(p, out, p->out.p, BN * sizeof(cplx), dev))) return e;
  if (p->timing) collect_timing(p, 2, 3, 1);
  p->ckptEvery = K;
  p->nSeg = nSeg;
  p->gInTime = in_time;
  p->bRows = rows;
  p->adjGen = ++p->gen;
  return NLM_OK;
}

static int batch_adjoint(nlm_plan* p, const double* g_out, double* g_in, bool dev);

extern "C" int nlm_batch_adjoint(nlm_plan* p, const double* g_out, double* g_in) {
  return batch_adjoint(p, g_out, g_in, false);
}

extern "C" int nlm_batch_adjoint_dev(nlm_plan* p, const double* g_out_dev, double* g_in_dev) {
  if (int e = check_device(p, g_out_dev, g_in_dev)) return e;
  return batch_adjoint(p, g_out_dev, g_in_dev, true);
}

static int batch_adjoint(nlm_plan* p, const double* g_out, double* g_in, bool dev) {
  if (int e = gnlse_diff_check(p)) return e;
  if (!g_out || !g_in) return set_err(NLM_INVALID_ARGUMENT, "null argument");
  if (p->bRows <= 0 || !p->nSeg || !p->ckpt.p)
    return set_err(NLM_RUNTIME_ERROR, "run nlm_batch_forward before the adjoint");
  if (p->adjGen != p->gen)
    return set_err(NLM_RUNTIME_ERROR,
                   "the medium changed after nlm_batch_forward (coefficients or another run); run the forward again "
                   "before the adjoint");
  const int N = p->N, nSteps = p->nZ - 1, rows = p->bRows, K = p->ckptEvery, nSeg = p->nSeg;
  const size_t BN = (size_t)rows * N;
  const Stager sg = pick_stager(p->L);
  int e;
  if ((e = p->gG.ensure(BN)) || (e = p->gtmp.ensure(BN)) || (e = p->adjWork.ensure(3 * BN)) ||
      (e = p->adjSeg.ensure((size_t)(p->ramanReal ? 6 : 8) * K * BN)))
    return e;
  if (dev) HIP_TRY(hipMemcpyAsync(p->gG.p, g_out, BN * sizeof(cplx), hipMemcpyDeviceToDevice, p->stream));
  else if ((e = nlm_to_device(p->gG.p, g_out, BN * sizeof(cplx), p->stream))) return e;
  BigParams bp;
  if ((e = setup_params(p, sg, rows, bp))) return e;
  bp.inCols = N;
  bp.nOut = 1;
  bp.outTime = p->gInTime;
  bp.ckpt = p->ckpt.p;
  bp.ckptEvery = K;
  bp.nSeg = nSeg;
  bp.seg = p->adjSeg.p;
  bp.GP = p->adjWork.p;
  bp.GA = bp.GP + BN;
  bp.TMP = bp.GA + BN;
  bp.gout = p->gG.p;
  bp.gin = p->gtmp.p;
  tic(p, 2);
  for (int s = nSeg - 1; s >= 0; s--) {
    const int i0 = s * K, i1 = i0 + K < nSteps ? i0 + K : nSteps;
    // recompute the segment from its checkpoint, keeping the stage data
    bp.segFirst = i0;
    bp.segLast = i1;
    sg.conv(bp, CV_RESUME, 0, 0, i0, p->stream);
    sg.mix(bp, MIX_STATE, 0, i0, p->stream);
    for (int i = i0 + 1; i <= i1; i++) launch_step(sg, bp, 0, i, p->stream, i == i1);
    launch_adjoint_segment(sg, bp, i0, i1, p->stream);
  }
  // the prologue a_0 = IFFT(halfIn FFT(in)) (time input) or IFFT(halfIn in)
  if (p->gInTime) {
    sg.conv(bp, CV_ADJ_OUT_TIME, 0, 0, 0, p->stream);
    sg.mix(bp, MIX_ADJ_OUT, 0, 0, p->stream);
  } else {
    sg.conv(bp, CV_ADJ_OUT_FREQ, 0, 0, 0, p->stream);
  }
  HIP_TRY(hipGetLastError());
  tic(p, 3);
  if ((e = from_device(p, g_in, p->gtmp.p, BN * sizeof(cplx), dev))) return e;
  if (p->timing) collect_timing(p, 2, 3, 1);
  return NLM_OK;
}
