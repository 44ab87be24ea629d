// nlm_mix.hpp -- in-register split step for even nFreqs that are not powers of two.
//
// A length N = R * (m_1 m_2 ...) * R with small factors is transformed by the same
// decimation-in-frequency scheme as nlm_fft.hpp: a field is held by T = N/R lanes,
// R points per lane in the stride layout (lane j holds x[j + T k], k < R).  Stage 0
// is a radix-R butterfly on the lane's own points, each middle stage (radices
// m_1, m_2, ..., run-time values) reads its butterflies from LDS and writes them
// back, and the last stage, radix R again, reads R adjacent points and leaves the
// result in the stride layout.  The first and last radix being equal, both
// directions take and return the same layout, so the pointwise work (RK4 stages,
// dispersion phase, impulses) stays in registers and a transform costs one LDS
// round trip per stage boundary.  R is a template parameter (register arrays), the
// middle radices and N are kernel arguments.
//
// Every signal mode of a medium has lanes of its own (nlm_modes.hpp).
//
// What bounds it: a wave's FP64 instructions (4 cycles each) and its 16-byte LDS accesses
// (~30 cycles each when nothing else runs on the SIMD), 70 % of its cycles at N = 600 by the
// counters, and the table reads, index arithmetic and stores between them.  nlm_any.hip's
// general kernel, which this replaces for these lengths, forms one output element per lane
// and pass: R table twiddles, R LDS reads and R complex products for every element instead
// of one butterfly per R elements.
// Measured, kernel ms before -> now: Chi2PDC Green's function N = 600, nZ = 200
// (1200 fields, 10 x 6 x 10, one wave each) 9.16 -> 1.41; in the same launch R = 5
// takes 2.41 and R = 2 3.69, while one field alone takes 1.15 (R = 5), 1.13 (R = 2)
// and 0.95 (R = 10) ms.  Other lengths at nZ = 200, first radix by mix_plan: Chi2PDC
// N = 144, one field 0.63 ms (R = 4; 0.70 with 6, 0.80 with 2); Chi2SHG N = 1000, 100 rows
// 1.63 ms.
#pragma once
#include <algorithm>
#include <cmath>

#include "nlm_modes.hpp"

constexpr int MIX_MAX_MID = 3;
constexpr int MIX_MAX_THREADS = 512;  // two waves per SIMD: 256 registers per lane

struct MixPlan {
  int N, R, T;         // T = N / R lanes hold one mode
  int TP;              // lanes from one group to the next
  int G;               // groups (signal modes)
  int FPB;             // fields per workgroup
  int threads;
  int waveFft;         // one group's lanes lie in one wave: its exchanges need no barrier
  int waveAll;         // the whole workgroup is one wave
  int bufElems;        // LDS elements per group
  int nMid;
  int mid[MIX_MAX_MID];
  unsigned magic[MIX_MAX_MID];  // ceil(2^32 / M) of the stage's sub-transform length M
  size_t ldsBytes;
  const cplx* tw;      // W_N^m
  double invN;
};

// q as a product of at most maxParts of `radices` (fewest parts first), or false.
inline bool mix_split(int q, int maxParts, int* parts, int* n) {
  static const int radices[] = {12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  *n = 0;
  if (q == 1) return true;
  for (int want = 1; want <= maxParts; want++)
    for (int r : radices) {
      if (q % r) continue;
      int rest = 0;
      if (want == 1 ? q != r : !mix_split(q / r, want - 1, parts + 1, &rest)) continue;
      parts[0] = r;
      *n = rest + 1;
      return true;
    }
  return false;
}

// Plan of the in-register mixed-radix kernels for `groups` modes of N points each and
// about `fields` independent fields; false if the length has none.  Every R with
// R^2 | N is tried with the fewest middle radices, and the one with the least
// estimated time is taken: a wave's points per stage (FP64 and LDS work) plus a
// latency per exchange (larger where its barrier joins several waves; fitted to
// the times above), times the rounds of waves that the fields make on the
// device's SIMDs (1024).  Few fields thus get more lanes and fewer points per lane, many
// fields the larger radices.
inline bool mix_plan(int N, int groups, long fields, bool gnlse, MixPlan* out) {
  static const int first[] = {10, 9, 8, 6, 5, 4, 3, 2};
  if (N < 8) return false;
  const double simds = 4.0 * device_cus();
  double best = 0;
  MixPlan p;
  for (int R : first) {
    if (N % (R * R) || (gnlse && R > 8)) continue;
    p = MixPlan{};
    if (!mix_split(N / (R * R), MIX_MAX_MID, p.mid, &p.nMid)) continue;
    p.N = N;
    p.R = R;
    p.T = N / R;
    p.G = groups;
    if (groups * p.T <= 64) {
      p.TP = p.T;
      p.FPB = 64 / (groups * p.T);
      p.threads = 64;
      p.waveFft = p.waveAll = 1;
    } else {
      p.TP = (p.T + 63) / 64 * 64;
      p.FPB = 1;
      p.threads = groups * p.TP;
      p.waveFft = p.TP == 64;
      p.waveAll = 0;
    }
    p.bufElems = N + p.T;  // rows of R points at pitch R + 1
    p.ldsBytes = ((size_t)N + (size_t)p.FPB * groups * p.bufElems) * sizeof(cplx);
    if (p.threads > MIX_MAX_THREADS || p.ldsBytes > 160 * 1024) continue;
    int P = R;
    double cost = 2.0 * R * (100 + 20 * std::log2((double)R));
    for (int s = 0; s < p.nMid; s++) {
      const int Q = p.mid[s], M = N / P / Q, it = (N / Q + p.TP - 1) / p.TP;
      p.magic[s] = M == 1 ? 0 : (unsigned)(((1ull << 32) + M - 1) / M);
      cost += it * Q * (130 + 20 * std::log2((double)Q));
      P *= Q;
    }
    cost += (p.waveFft ? 400.0 : 900.0) * (p.nMid + 1);
    const double waves = (double)((fields + p.FPB - 1) / p.FPB) * (p.threads / 64);
    cost *= std::max(1.0, waves / simds);
    if (best == 0 || cost < best) {
      best = cost;
      *out = p;
    }
  }
  if (best == 0) return false;
  out->invN = 1.0 / N;
  return true;
}

extern __shared__ cplx mix_lds[];

namespace mix {

using namespace modes;

// R-point DFT in place, natural order in and out; forward exp(-2 pi i nk/R).
template <int R, bool INV>
__device__ __forceinline__ void dft(cplx* v);

template <bool INV>
__device__ __forceinline__ void dft3(cplx& a, cplx& b, cplx& c) {
  constexpr double s = 0.86602540378443864676;  // sin(2 pi / 3)
  const cplx t = b + c, d = mul_mi<INV>(s * (b - c));
  const cplx m = a - 0.5 * t;
  a = a + t;
  b = m + d;
  c = m - d;
}

template <bool INV>
__device__ __forceinline__ void dft5(cplx& a, cplx& b, cplx& c, cplx& d, cplx& e) {
  constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;  // cos(2 pi/5), cos(4 pi/5)
  constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;   // sin(2 pi/5), sin(4 pi/5)
  const cplx t1 = b + e, t2 = c + d, t3 = b - e, t4 = c - d;
  const cplx m1 = a + c1 * t1 + c2 * t2, m2 = a + c2 * t1 + c1 * t2;
  const cplx n1 = mul_mi<INV>(s1 * t3 + s2 * t4), n2 = mul_mi<INV>(s2 * t3 - s1 * t4);
  a = a + t1 + t2;
  b = m1 + n1;
  e = m1 - n1;
  c = m2 + n2;
  d = m2 - n2;
}

template <bool INV>
__device__ __forceinline__ void dft7(cplx* v) {
  constexpr double c1 = 0.62348980185873353053, c2 = -0.22252093395631440429, c3 = -0.90096886790241912624;
  constexpr double s1 = 0.78183148246802980871, s2 = 0.97492791218182360702, s3 = 0.43388373911755812048;
  const cplx p1 = v[1] + v[6], p2 = v[2] + v[5], p3 = v[3] + v[4];
  const cplx q1 = v[1] - v[6], q2 = v[2] - v[5], q3 = v[3] - v[4];
  const cplx a = v[0];
  const cplx m1 = a + c1 * p1 + c2 * p2 + c3 * p3, m2 = a + c2 * p1 + c3 * p2 + c1 * p3,
             m3 = a + c3 * p1 + c1 * p2 + c2 * p3;
  const cplx n1 = mul_mi<INV>(s1 * q1 + s2 * q2 + s3 * q3), n2 = mul_mi<INV>(s2 * q1 - s3 * q2 - s1 * q3),
             n3 = mul_mi<INV>(s3 * q1 - s1 * q2 + s2 * q3);
  v[0] = a + p1 + p2 + p3;
  v[1] = m1 + n1;
  v[6] = m1 - n1;
  v[2] = m2 + n2;
  v[5] = m2 - n2;
  v[3] = m3 + n3;
  v[4] = m3 - n3;
}

// Coprime factors (Good-Thomas): input n = (B n1 + A n2) mod AB, output k with
// k = k1 mod A and k = k2 mod B; no twiddles.
template <int A, int B, bool INV>
__device__ __forceinline__ void dft_coprime(cplx* v) {
  constexpr int R = A * B;
  cplx x[A][B];
#pragma unroll
  for (int n1 = 0; n1 < A; n1++)
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) x[n1][n2] = v[(B * n1 + A * n2) % R];
#pragma unroll
  for (int n1 = 0; n1 < A; n1++) dft<B, INV>(x[n1]);
#pragma unroll
  for (int k2 = 0; k2 < B; k2++) {
    cplx y[A];
#pragma unroll
    for (int n1 = 0; n1 < A; n1++) y[n1] = x[n1][k2];
    dft<A, INV>(y);
#pragma unroll
    for (int n1 = 0; n1 < A; n1++) x[n1][k2] = y[n1];
  }
  // exp(-2 pi i k (B n1 + A n2)/AB) = exp(-2 pi i k n1/A) exp(-2 pi i k n2/B)
#pragma unroll
  for (int k = 0; k < R; k++) v[k] = x[k % A][k % B];
}

template <bool INV>
__device__ __forceinline__ void dft9(cplx* v) {
  // 9 = 3 x 3: n = 3 n1 + n2, k = k1 + 3 k2, twiddles W_9^(n2 k1)
  constexpr double w1r = 0.76604444311897803520, w1i = -0.64278760968653932632;   // W_9
  constexpr double w2r = 0.17364817766693034885, w2i = -0.98480775301220805937;   // W_9^2
  constexpr double w4r = -0.93969262078590838405, w4i = -0.34202014332566873304;  // W_9^4
#pragma unroll
  for (int n2 = 0; n2 < 3; n2++) dft3<INV>(v[n2], v[3 + n2], v[6 + n2]);
  v[4] = twmul<INV>(v[4], mk(w1r, w1i));
  v[5] = twmul<INV>(v[5], mk(w2r, w2i));
  v[7] = twmul<INV>(v[7], mk(w2r, w2i));
  v[8] = twmul<INV>(v[8], mk(w4r, w4i));
#pragma unroll
  for (int k1 = 0; k1 < 3; k1++) dft3<INV>(v[3 * k1], v[3 * k1 + 1], v[3 * k1 + 2]);
  // v[3 k1 + k2] is output k1 + 3 k2
  const cplx a = v[1], b = v[2], c = v[5];
  v[1] = v[3];
  v[3] = a;
  v[2] = v[6];
  v[6] = b;
  v[5] = v[7];
  v[7] = c;
}

template <int R, bool INV>
__device__ __forceinline__ void dft(cplx* v) {
  if constexpr (R == 2 || R == 4 || R == 8) dft_small<R, INV>(v);
  else if constexpr (R == 3) dft3<INV>(v[0], v[1], v[2]);
  else if constexpr (R == 5) dft5<INV>(v[0], v[1], v[2], v[3], v[4]);
  else if constexpr (R == 6) dft_coprime<2, 3, INV>(v);
  else if constexpr (R == 7) dft7<INV>(v);
  else if constexpr (R == 9) dft9<INV>(v);
  else if constexpr (R == 10) dft_coprime<2, 5, INV>(v);
  else if constexpr (R == 12) dft_coprime<4, 3, INV>(v);
}

// One group's view of its field: lane j of the T that hold a mode, its LDS buffer
// and the first stage's twiddles W_N^(j c).
template <int RADIX>
struct Fft {
  static constexpr int R = RADIX;
  const MixPlan& p;
  cplx* buf;
  const cplx* tab;  // LDS copy of W_N^m
  int j;
  bool on;          // j < T
  // from R = 9 the first twiddles are read from the table at use: in registers they
  // spilled beside the step matrices
  static constexpr bool W0_REG = R <= 8;
  cplx w0[W0_REG ? R : 1];

  __device__ __forceinline__ Fft(const MixPlan& p_, cplx* b, const cplx* t, int j_) : p(p_), buf(b), tab(t), j(j_) {
    on = j < p.T;
    if constexpr (W0_REG)
#pragma unroll
      for (int c = 1; c < R; c++) w0[c] = tab[on ? j * c : 0];
  }

  __device__ __forceinline__ int at(int k) const { return j + p.T * k; }
  __device__ __forceinline__ int n() const { return p.N; }
  __device__ __forceinline__ double invN() const { return p.invN; }
  __device__ __forceinline__ int bufElems() const { return p.bufElems; }
  __device__ __forceinline__ void sync() const { sync_if(p.waveFft); }
  __device__ __forceinline__ void syncAll() const { sync_if(p.waveAll); }

  // Middle stage of radix Q: butterflies beta = j, j + TP, ... read [g][a][b]
  // (sub-arrays g of Q M points), write [g + P c][b]; `pitch` is the written
  // sub-array's row length (M, or the padded M before the last stage).
  template <int Q, bool INV>
  __device__ __forceinline__ void middle(int P, int M, unsigned magic, int pitch) {
    // P before, M after this stage: N = P Q M.  A lane holds at most as many points
    // as the stride layout gives it, rounded up to whole butterflies.
    constexpr int IT = (R + Q - 1) / Q;
    const int nb = p.N / Q;
    cplx x[IT][Q];
    int bb[IT], gg[IT];
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const int beta = j + i * p.TP;
      const int g = M == 1 ? beta : (int)__umulhi((unsigned)beta, magic);
      const int b = beta - g * M;
      bb[i] = b;
      gg[i] = g;
      if (beta < nb)
#pragma unroll
        for (int a = 0; a < Q; a++) x[i][a] = buf[g * Q * M + a * M + b];
    }
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const int beta = j + i * p.TP;
      if (beta < nb) {
        dft<Q, INV>(x[i]);
#pragma unroll
        for (int c = 1; c < Q; c++) x[i][c] = twmul<INV>(x[i][c], tab[bb[i] * c * P]);
      }
    }
    sync();  // every reader of the previous layout is done
#pragma unroll
    for (int i = 0; i < IT; i++) {
      const int beta = j + i * p.TP;
      if (beta < nb)
#pragma unroll
        for (int c = 0; c < Q; c++) buf[(gg[i] + P * c) * pitch + bb[i]] = x[i][c];
    }
  }

  // Transform v (stride layout in and out); inverse unscaled.  `fetch` runs before
  // the last exchange's reads: loads issued there are covered by the last stage
  // without their registers being live through the middle ones.
  template <bool INV, class Fetch>
  __device__ __forceinline__ void run(cplx (&v)[R], Fetch&& fetch) {
    // rows of R points before the last stage are stored with an odd pitch, so that
    // its reads of R adjacent points per lane spread over the banks
    constexpr int RP = R | 1;
    // LDS offsets are formed here, not hoisted out of the z loop for every middle
    // radix, where they spilled
    j = opaque_lane(j);
    dft<R, INV>(v);
#pragma unroll
    for (int c = 1; c < R; c++) {
      if constexpr (W0_REG) v[c] = twmul<INV>(v[c], w0[c]);
      else v[c] = twmul<INV>(v[c], tab[on ? j * c : 0]);
    }
    sync();  // previous readers of buf are done
    {
      const int row = p.nMid == 0 ? RP : p.T;
      if (on)
#pragma unroll
        for (int c = 0; c < R; c++) buf[c * row + j] = v[c];
    }
    int P = R;
    for (int s = 0; s < p.nMid; s++) {
      const int Q = p.mid[s], M = p.N / P / Q;
      const int pitch = s == p.nMid - 1 ? RP : M;
      const unsigned mg = p.magic[s];
      sync();
      switch (Q) {
        case 2: middle<2, INV>(P, M, mg, pitch); break;
        case 3: middle<3, INV>(P, M, mg, pitch); break;
        case 4: middle<4, INV>(P, M, mg, pitch); break;
        case 5: middle<5, INV>(P, M, mg, pitch); break;
        case 6: middle<6, INV>(P, M, mg, pitch); break;
        case 7: middle<7, INV>(P, M, mg, pitch); break;
        case 8: middle<8, INV>(P, M, mg, pitch); break;
        case 9: middle<9, INV>(P, M, mg, pitch); break;
        case 10: middle<10, INV>(P, M, mg, pitch); break;
        default: middle<12, INV>(P, M, mg, pitch); break;
      }
      P *= Q;
    }
    fetch();
    sync();
    if (on)
#pragma unroll
      for (int a = 0; a < R; a++) v[a] = buf[j * RP + a];
    dft<R, INV>(v);
  }
  template <bool INV>
  __device__ __forceinline__ void run(cplx (&v)[R]) {
    run<INV>(v, [] {});
  }
};

// The lane's place in the workgroup: field slot, group and lane within the group.
struct Place {
  int slot, g, j;
};
__device__ __forceinline__ Place place(const MixPlan& p) {
  Place a;
  const int lpf = p.G * p.TP;  // lanes per field
  if (p.FPB == 1) {
    a.slot = 0;
    a.g = threadIdx.x / p.TP;
    a.j = threadIdx.x - a.g * p.TP;
    if (p.TP % 64 == 0) {
      a.g = __builtin_amdgcn_readfirstlane(a.g);  // a group is whole waves
    } else if (a.g >= p.G) {  // one field's groups in one wave: its spare lanes
      a.g = 0;
      a.j = 1 << 20;
    }
  } else {
    a.slot = threadIdx.x / lpf;
    const int r = threadIdx.x - a.slot * lpf;
    a.g = r / p.TP;
    a.j = r - a.g * p.TP;
    if (a.slot >= p.FPB) {  // lanes past the last field: no points and no butterflies
      a.slot = p.FPB - 1;
      a.g = 0;
      a.j = 1 << 20;
    }
  }
  return a;
}

// Copy the twiddle table into LDS (all threads; ends with a barrier); returns it.
__device__ __forceinline__ const cplx* load_table(const MixPlan& p, cplx* lds) {
  for (int k = threadIdx.x; k < p.N; k += blockDim.x) lds[k] = p.tw[k];
  __syncthreads();
  return lds;
}

// A one-mode medium whose RK4 step is the real 2x2 matrix of kp.tab (see
// nlm_prop_tab.hip; the table holds the inverse transform's 1/N).
struct Table {
  static constexpr int NS = 1;
};

template <int R>
__device__ __forceinline__ void get_matrices(const Fft<R>& f, cplx (&al)[R], cplx (&be)[R],
                                             const cplx* __restrict__ row) {
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int i = f.on ? f.at(k) : 0;
    al[k] = row[(size_t)i * 2];
    be[k] = row[(size_t)i * 2 + 1];
  }
}

template <int R>
__device__ __forceinline__ void table_field(const KParams& kp, Fft<R>& f, int field, bool act) {
  const int N = f.p.N;
  cplx v[R];
  enter<1>(kp, f, field, 0, act, v);
  cplx al[R], be[R];
  if (kp.nZ > 1) {
    f.template run<true>(v);
    if (kp.kind == KIND_GRID) put_scaled(f, grid_row(kp, kp.gridT, field, 1, 0, 0, N), v, act);
    get_matrices<R>(f, al, be, kp.tab + (size_t)N * 2);
  }
  for (int i = 1; i < kp.nZ; i++) {
#pragma unroll
    for (int k = 0; k < R; k++) {
      const cplx x = v[k];
      v[k] = mk(al[k].re * x.re + al[k].im * x.im, be[k].re * x.re + be[k].im * x.im);
    }
    f.template run<false>(v);
    mul_row(f, v, kp.dstep);
    if (i < kp.nZ - 1) {
      if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridF, field, 1, 0, i, N), v, act);
      f.template run<true>(v, [&]() __attribute__((always_inline)) { get_matrices<R>(f, al, be, kp.tab + (size_t)(i + 1) * N * 2); });
      if (kp.kind == KIND_GRID) put_scaled(f, grid_row(kp, kp.gridT, field, 1, 0, i, N), v, act);
    }
  }
  leave<1>(kp, f, field, 0, act, v);
}

// One Chi3GNLSE field (solvers/Chi3GNLSE.cpp:51-92), state and RK4 sum kept as spectra as in
// the power-of-two kernel (16 transforms per step): FFT(k) of a stage is
// filter FFT( IFFT(FFT(r |y|^2) R) y ).
template <int R>
__device__ __forceinline__ void gnlse_field(const KParams& kp, Fft<R>& f, int field, bool act) {
  const int N = f.p.N;
  cplx v[R], y[R];  // v: spectrum; y: time-domain stage input
  enter<1>(kp, f, field, 0, act, v);
  if (kp.nZ > 1) {
#pragma unroll
    for (int m = 0; m < R; m++) y[m] = v[m];
    f.template run<true>(y);
    scale_row(f, y);
    if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridT, field, 1, 0, 0, N), y, act);
  }
  for (int i = 1; i < kp.nZ; i++) {
    const uniform_cplx* c = to_uniform(kp.coef + (size_t)i * 3);
    // acc accumulates ((k1 + 2 k2) + 2 k3) + k4 in the reference's order
    cplx acc[R];
#pragma unroll
    for (int m = 0; m < R; m++) acc[m] = mk(0.0, 0.0);
    // one copy of the four transforms for the four stages
#pragma unroll 1
    for (int s = 0; s < 4; s++) {
      const double r = s == 0 ? c[0].re : s == 3 ? c[2].re : c[1].re;
      cplx k[R];
#pragma unroll
      for (int m = 0; m < R; m++) k[m] = mk(r * abs2(y[m]), 0.0);
      f.template run<false>(k);
      mul_row(f, k, kp.raman);
      f.template run<true>(k);
      scale_row(f, k);
#pragma unroll
      for (int m = 0; m < R; m++) k[m] = k[m] * y[m];
      f.template run<false>(k);
      mul_row(f, k, kp.filt);
      const double wa = s == 1 || s == 2 ? 2.0 : 1.0, wy = s == 2 ? 1.0 : 0.5;
#pragma unroll
      for (int m = 0; m < R; m++) acc[m] = acc[m] + wa * k[m];
      if (s < 3) {
#pragma unroll
        for (int m = 0; m < R; m++) y[m] = v[m] + wy * k[m];
      } else {
#pragma unroll
        for (int m = 0; m < R; m++) v[m] = v[m] + acc[m] * (1. / 6.);
        mul_row(f, v, kp.dstep);
        if (i == kp.nZ - 1) break;
        if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridF, field, 1, 0, i, N), v, act);
#pragma unroll
        for (int m = 0; m < R; m++) y[m] = v[m];
      }
      f.template run<true>(y);
      scale_row(f, y);
    }
    if (i < kp.nZ - 1 && kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridT, field, 1, 0, i, N), y, act);
  }
  leave<1>(kp, f, field, 0, act, v);
}

}  // namespace mix

// One workgroup per FPB fields; LDS: the twiddle table, then G buffers per field.
template <class M, int R>
__global__ void __launch_bounds__(MIX_MAX_THREADS) k_mix_prop(KParams kp, MixPlan p) {
  const cplx* tab = mix::load_table(p, mix_lds);
  const mix::Place a = mix::place(p);
  cplx* fieldBuf = mix_lds + p.N + (size_t)a.slot * p.G * p.bufElems;
  mix::Fft<R> f(p, fieldBuf + a.g * p.bufElems, tab, a.j);
  const int field = blockIdx.x * p.FPB + a.slot;
  const bool act = f.on && field < kp.nFields;
  if constexpr (std::is_same<M, mix::Table>::value) mix::table_field<R>(kp, f, field, act);
  else if constexpr (std::is_same<M, MChi3GNLSE>::value) mix::gnlse_field<R>(kp, f, field, act);
  else modes::modes_field<M>(kp, f, fieldBuf, field, a.g, act);
}

typedef void (*mix_fn)(const KParams&, const MixPlan&, int grid, hipStream_t);

template <class M, int R>
void launch_mix_prop(const KParams& kp, const MixPlan& p, int grid, hipStream_t s) {
  hipLaunchKernelGGL((k_mix_prop<M, R>), dim3(grid), dim3(p.threads), p.ldsBytes, s, kp, p);
}

// Launchers per solver (nlm_mix_inst.hip; Chi3 and Chi2PDC through their step table,
// Chi2AFC as Chi2SFG, Chi2ASHG as Chi2SHG) and of the row kernels (nlm_mix_rows.hip);
// nullptr where R is not built.
mix_fn nlm_pick_mix_1(int R), nlm_pick_mix_2(int R), nlm_pick_mix_4(int R), nlm_pick_mix_5(int R),
    nlm_pick_mix_6(int R), nlm_pick_mix_7(int R), nlm_pick_mix_8(int R), nlm_pick_mix_9(int R),
    nlm_pick_mix_10(int R), nlm_pick_mix_11(int R), nlm_pick_mix_12(int R), nlm_pick_mix_14(int R);

struct MixRows {
  const cplx* in;       // transforms: rows in and out
  cplx* out;
  int count, inverse;
  const cplx* F0;       // pumps
  const cplx* env;
  const double* Dp;
  double dzp;
  const double* strength;
  const cplx* dstepP;
  const cplx* relI;
  int nZP;
  cplx* pumpF;
  cplx* pumpT;
};
enum { MIX_ROWS_FFT = 0, MIX_ROWS_LINEAR = 1, MIX_ROWS_CHI3 = 2 };
// false where plan.R is not built
bool nlm_mix_rows(int kind, const MixRows& r, const MixPlan& p, hipStream_t s);
