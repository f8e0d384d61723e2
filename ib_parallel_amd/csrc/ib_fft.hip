// ib_fft.hip -- unnormalised 2-D DST-I (FFTW RODFT00 x RODFT00) on CDNA4.
//
// Replaces the FFTW-MPI transforms of src/myfft.F90:168-213.  A 2-D DST is a
// row (x) pass and a column (y) pass.  Each pass evaluates two real DST-I of
// length N at once with one complex FFT of length L = 2(N+1): the pair
// (x_a, x_b) is packed as z = x_a + i x_b and extended oddly
// (z_0 = z_M = 0, z_{2M-t} = -z_t), then
//     Z = -2i S(x_a) + 2 S(x_b)   =>   S(x_a) = -Im Z,  S(x_b) = Re Z.
// The FFT is a mixed-radix Stockham autosort run entirely in LDS with two
// ping-pong buffers per transform: radix 4/2/3/5 butterflies live in
// registers, any larger prime factor uses one thread per output.  Fused
// pre/post operations keep the ctci/ainv/predictor spectral products inside
// the column pass (Y_SCALE2, Y_PRED) and apply_bc / the corrector subtraction
// inside the row pass (X_APPLYBC, X_SUBFROM).
#include <array>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "ib_device.h"
#include "ib_kernels.h"

namespace ibg {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

template <int R>
__device__ __forceinline__ void dft(double2* v);

template <>
__device__ __forceinline__ void dft<2>(double2* v) {
  double2 a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <>
__device__ __forceinline__ void dft<3>(double2* v) {
  const double s3 = 0.86602540378443864676;  // sin(2 pi / 3)
  double2 t = cadd(v[1], v[2]), d = csub(v[1], v[2]);
  double2 mm = make_double2(v[0].x - 0.5 * t.x, v[0].y - 0.5 * t.y);
  double2 jd = make_double2(s3 * d.y, -s3 * d.x);  // -i s3 d
  v[0] = cadd(v[0], t);
  v[1] = cadd(mm, jd);
  v[2] = csub(mm, jd);
}

template <>
__device__ __forceinline__ void dft<4>(double2* v) {
  double2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
  double2 c = cadd(v[1], v[3]), d = csub(v[1], v[3]);
  v[0] = cadd(a, c);
  v[2] = csub(a, c);
  v[1] = make_double2(b.x + d.y, b.y - d.x);  // b - i d
  v[3] = make_double2(b.x - d.y, b.y + d.x);  // b + i d
}

template <>
__device__ __forceinline__ void dft<5>(double2* v) {
  const double c1 = 0.30901699437494742410;   // cos(2 pi/5)
  const double c2 = -0.80901699437494742410;  // cos(4 pi/5)
  const double s1 = 0.95105651629515357212;   // sin(2 pi/5)
  const double s2 = 0.58778525229247312917;   // sin(4 pi/5)
  double2 p1 = cadd(v[1], v[4]), m1 = csub(v[1], v[4]);
  double2 p2 = cadd(v[2], v[3]), m2 = csub(v[2], v[3]);
  double2 a1 = make_double2(v[0].x + c1 * p1.x + c2 * p2.x, v[0].y + c1 * p1.y + c2 * p2.y);
  double2 a2 = make_double2(v[0].x + c2 * p1.x + c1 * p2.x, v[0].y + c2 * p1.y + c1 * p2.y);
  double2 b1 = make_double2(s1 * m1.x + s2 * m2.x, s1 * m1.y + s2 * m2.y);
  double2 b2 = make_double2(s2 * m1.x - s1 * m2.x, s2 * m1.y - s1 * m2.y);
  v[0] = make_double2(v[0].x + p1.x + p2.x, v[0].y + p1.y + p2.y);
  v[1] = make_double2(a1.x + b1.y, a1.y - b1.x);  // a1 - i b1
  v[4] = make_double2(a1.x - b1.y, a1.y + b1.x);  // a1 + i b1
  v[2] = make_double2(a2.x + b2.y, a2.y - b2.x);  // a2 - i b2
  v[3] = make_double2(a2.x - b2.y, a2.y + b2.x);  // a2 + i b2
}

template <>
__device__ __forceinline__ void dft<8>(double2* v) {
  const double c = 0.70710678118654752440;  // cos(pi/4)
  double2 e[4] = {v[0], v[2], v[4], v[6]};
  double2 o[4] = {v[1], v[3], v[5], v[7]};
  dft<4>(e);
  dft<4>(o);
  // o[k] *= exp(-2 pi i k / 8)
  const double2 o1 = make_double2(c * (o[1].x + o[1].y), c * (o[1].y - o[1].x));
  const double2 o2 = make_double2(o[2].y, -o[2].x);
  const double2 o3 = make_double2(c * (o[3].y - o[3].x), -c * (o[3].x + o[3].y));
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[5] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[6] = csub(e[2], o2);
  v[3] = cadd(e[3], o3);
  v[7] = csub(e[3], o3);
}

// One Stockham stage of radix R over nf transforms of length L stored at
// in[s*L + t]; Ns = product of the radices already applied.
template <int R>
__device__ __forceinline__ void stage_fixed(const double2* __restrict__ in, double2* __restrict__ out, int nf,
                                            int L, int Ns, const double2* __restrict__ W) {
  const int LR = L / R;
  const int tws = LR / Ns;
  const int total = nf * LR;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int s = idx / LR;
    const int j = idx - s * LR;
    const double2* ip = in + s * L;
    double2* op = out + s * L;
    const int k = j % Ns;
    double2 v[R];
    v[0] = ip[j];
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul(ip[j + r * LR], W[k * r * tws]);
    dft<R>(v);
    const int base = (j - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) op[base + r * Ns] = v[r];
  }
}

// A stage of any other radix R (an odd prime >= 7) as a direct length-R DFT
// using its conjugate symmetry.  Pass 1 applies the inter-stage twiddles and
// folds each input pair in place: p_r = x_r + x_(R-r) at position r and
// m_r = x_r - x_(R-r) at position R-r (r = 1..H, H = (R-1)/2).  Pass 2 forms
// U_q = sum p_r cos(2 pi rq/R) and V_q = sum m_r sin(2 pi rq/R), which give
// both X_q = x_0 + U_q - i V_q and X_(R-q) = x_0 + U_q + i V_q: a quarter of
// the real products of the plain sum.  Each thread holds a tile of 2
// sub-transforms x 4 values of q, so every LDS read feeds several products.
// lanes one transform's tiles of the generic stage may spread over (the
// threads of a one-transform workgroup)
constexpr int kGenSplitLanes = 256;

__device__ void stage_generic(double2* __restrict__ in, double2* __restrict__ out, int nf, int L, int Ns, int R,
                              const double2* __restrict__ W) {
  const int LR = L / R;
  const int tws = LR / Ns;
  const int H = (R - 1) / 2;
  for (int idx = threadIdx.x; idx < nf * LR * H; idx += blockDim.x) {
    const int s = idx / (LR * H);
    const int u = idx - s * (LR * H);
    const int r = 1 + u / LR, j = u % LR;
    double2* x = in + s * L + j;
    double2 xa = x[r * LR], xb = x[(R - r) * LR];
    const int k = j % Ns;
    if (k) {
      xa = cmul(xa, W[k * r * tws]);
      xb = cmul(xb, W[k * (R - r) * tws]);
    }
    x[r * LR] = cadd(xa, xb);
    x[(R - r) * LR] = csub(xa, xb);
  }
  __syncthreads();
  const int nj = (LR + 1) / 2, nq = (H + 4) / 4;  // q = 0..H in groups of 4
  const int ntile = nf * nj * nq;
  // with few tiles per transform, 2 or 4 adjacent lanes share a tile's sum
  // over r (terms r = 1 + part, 1 + part + split, ...) and combine it by
  // lane shuffles.  The split depends on the transform's own tile count
  // only (not on how many transforms share the workgroup, nor on its size),
  // so every tile shape of the DST passes sums in the same order and gives
  // the same bits.
  int lsplit = 0;
  while (lsplit < 2 && ((nj * nq) << (lsplit + 1)) <= kGenSplitLanes) ++lsplit;
  const int split = 1 << lsplit;
  for (int tt = threadIdx.x; tt < (ntile << lsplit); tt += blockDim.x) {
    const int t = tt >> lsplit, part = tt & (split - 1);
    const int s = t / (nj * nq);
    const int u = t - s * (nj * nq);
    const int qt = u / nj;
    const int j0 = 2 * (u - qt * nj), q0 = 4 * qt;
    const int j1 = min(j0 + 1, LR - 1);  // an odd LR repeats the last column (not stored)
    const double2* __restrict__ x = in + s * L;
    // cos/sin of 2 pi rq/R from W[((r q) mod R) LR] = (cos, -sin), the index
    // kept running below L per value of q
    int bq[4], dq[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int qL = min(q0 + c, H) * LR;  // below L
      bq[c] = (int)(((long)(1 + part) * qL) % L);
      dq[c] = (int)(((long)split * qL) % L);
    }
    double2 U0[4], V0[4], U1[4], V1[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) U0[c] = V0[c] = U1[c] = V1[c] = make_double2(0.0, 0.0);
    for (int r = 1 + part; r <= H; r += split) {
      const double2 pa = x[j0 + r * LR], ma = x[j0 + (R - r) * LR];
      const double2 pb = x[j1 + r * LR], mb = x[j1 + (R - r) * LR];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double2 w = W[bq[c]];
        const double cs = w.x, sn = -w.y;
        U0[c] = make_double2(U0[c].x + pa.x * cs, U0[c].y + pa.y * cs);
        V0[c] = make_double2(V0[c].x + ma.x * sn, V0[c].y + ma.y * sn);
        U1[c] = make_double2(U1[c].x + pb.x * cs, U1[c].y + pb.y * cs);
        V1[c] = make_double2(V1[c].x + mb.x * sn, V1[c].y + mb.y * sn);
        bq[c] += dq[c];
        if (bq[c] >= L) bq[c] -= L;
      }
    }
    for (int off = 1; off < split; off <<= 1) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        U0[c].x += __shfl_xor(U0[c].x, off); U0[c].y += __shfl_xor(U0[c].y, off);
        V0[c].x += __shfl_xor(V0[c].x, off); V0[c].y += __shfl_xor(V0[c].y, off);
        U1[c].x += __shfl_xor(U1[c].x, off); U1[c].y += __shfl_xor(U1[c].y, off);
        V1[c].x += __shfl_xor(V1[c].x, off); V1[c].y += __shfl_xor(V1[c].y, off);
      }
    }
    if (part) continue;
    const double2 x0a = x[j0], x0b = x[j1];
    double2* __restrict__ o = out + s * L;
    const int k0 = j0 % Ns, k1 = (j0 + 1) % Ns;
    const bool second = j0 + 1 < LR;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int q = q0 + c;
      if (q <= H) {
        const int ba = (j0 - k0) * R + k0, bb = (j0 + 1 - k1) * R + k1;
        o[ba + q * Ns] = make_double2(x0a.x + U0[c].x + V0[c].y, x0a.y + U0[c].y - V0[c].x);
        if (second) o[bb + q * Ns] = make_double2(x0b.x + U1[c].x + V1[c].y, x0b.y + U1[c].y - V1[c].x);
        if (q > 0) {
          o[ba + (R - q) * Ns] = make_double2(x0a.x + U0[c].x - V0[c].y, x0a.y + U0[c].y + V0[c].x);
          if (second) o[bb + (R - q) * Ns] = make_double2(x0b.x + U1[c].x - V1[c].y, x0b.y + U1[c].y + V1[c].x);
        }
      }
    }
  }
}

// Runs the plan on nf transforms held in a (scratch b) with the twiddle table
// W staged in LDS; returns the buffer that holds the result.  Caller
// synchronises before the call.  GEN = false leaves out the stage of radix
// >= 7 (stage_generic, whose registers set the kernel's occupancy): the host
// launches that form only for plans whose radices are all 2, 3, 4, 5, 8.
// Only the row pass has it: the column pass built without the stage
// measured slower (its two-input form 23.4 against 16.7 us per launch at
// 400 x 400, the same LDS-bound occupancy), so it always keeps the stage.
template <bool GEN>
__device__ __forceinline__ double2* fft_run(double2* a, double2* b, int nf, const FFTPlan& pl, const double2* W) {
  int Ns = 1;
  for (int st = 0; st < pl.nst; ++st) {
    const int R = pl.rad[st];
    switch (R) {
      case 8: stage_fixed<8>(a, b, nf, pl.L, Ns, W); break;
      case 4: stage_fixed<4>(a, b, nf, pl.L, Ns, W); break;
      case 2: stage_fixed<2>(a, b, nf, pl.L, Ns, W); break;
      case 3: stage_fixed<3>(a, b, nf, pl.L, Ns, W); break;
      case 5: stage_fixed<5>(a, b, nf, pl.L, Ns, W); break;
      default:
        if constexpr (GEN) {
          stage_generic(a, b, nf, pl.L, Ns, R, W);
        } else {
          // a plan this form cannot run (the host never launches one): the
          // result is NaN, never a stale buffer
          for (int i = threadIdx.x; i < nf * pl.L; i += blockDim.x) b[i] = make_double2(__builtin_nan(""), __builtin_nan(""));
        }
        break;
    }
    __syncthreads();
    double2* t = a;
    a = b;
    b = t;
    Ns *= R;
  }
  return a;
}


// X_POINTROT: rot(E^T e_k) at node (i, j), formed from the 49 taps of force
// entry k (the x-face or y-face patch centred on (ix, iy)); with no weights,
// rot of the unit face source at (ix, iy).
struct PointPatch {
  int comp, ix, iy;
  const double* w;
  __device__ double face(int c, int i, int j) const {
    if (c != comp) return 0.0;
    const int p = i - ix, l = j - iy;
    if (!w) return (p == 0 && l == 0) ? 1.0 : 0.0;
    if (p < -3 || p > 3 || l < -3 || l > 3) return 0.0;
    return w[(l + 3) * 7 + (p + 3)];
  }
  __device__ double rot(int i, int j) const {
    return face(2, i, j) - face(2, i - 1, j) - face(1, i, j) + face(1, i, j - 1);
  }
};


// Stage the twiddle table in LDS (read by every stage of every transform).
__device__ __forceinline__ void load_twiddles(double2* Wl, const FFTPlan& pl) {
  for (int t = threadIdx.x; t < pl.L; t += blockDim.x) Wl[t] = pl.W[t];
}

// X_POINTROT: the patch of batch element by; false when this workgroup's rows
// see no tap: they transform to zero, which is written
__device__ __forceinline__ bool point_rows(const XArgs& a, PointPatch& pt, int by, int pair0, double* out) {
  const int k = a.c0 + by;
  // centre tap (p = l = 0) of force entry k, or face k of a face list
  const int ck = a.w ? a.key[k * kTaps + kTaps / 2] : a.key[k];
  const Geom& g = a.g;
  const int N = a.pl.N, rp = a.rp, nrows = g.n - 1;
  if (ck < g.Fx) { pt.comp = 1; pt.ix = ck % (g.m + 1) + 1; pt.iy = ck / (g.m + 1) + 1; }
  else { pt.comp = 2; pt.ix = (ck - g.Fx) % g.m + 1; pt.iy = (ck - g.Fx) / g.m + 1; }
  pt.w = a.w ? a.w + (long)k * kTaps : nullptr;
  const int j0 = 2 * pair0 + 2, j1 = 2 * (pair0 + rp) + 1;  // node rows of this workgroup
  if (j1 >= pt.iy - 3 && j0 <= pt.iy + 4) return true;
  for (int idx = threadIdx.x; idx < rp * N; idx += blockDim.x) {
    const int s = idx / N, t = idx - s * N;
    const int ra = 2 * (pair0 + s), rb = ra + 1;
    if (ra < nrows) out[(long)ra * N + t] = 0.0;
    if (rb < nrows) out[(long)rb * N + t] = 0.0;
  }
  return false;
}

// The row pass's input at node (i, j).
template <int MODE>
__device__ __forceinline__ double row_value(const XArgs& a, const PointPatch& pt, const double* __restrict__ in,
                                            const double* __restrict__ bc, int i, int j) {
  const Geom& g = a.g;
  double x;
  if (MODE == X_POINTROT) {
    x = pt.rot(i, j);
  } else if (MODE == X_ROT) {
    // rot_int + rot_bc: vort(i,j) = hy(i,j) - hy(i-1,j) - hx(i,j) + hx(i,j-1)
    x = a.hy[(i - 1) + g.m * (j - 1)] - a.hy[(i - 2) + g.m * (j - 1)] - a.hx[(i - 1) + (g.m + 1) * (j - 1)] +
        a.hx[(i - 1) + (g.m + 1) * (j - 2)];
  } else {
    x = in[(long)(j - 2) * (g.m - 1) + (i - 2)];
  }
  if (MODE == X_APPLYBC) {
    // apply_bc(vort, sbc, 1.d0), src/operators_fluid.F90:539-549
    if (i == 2) x = x + bc[g.left + j - 1];
    if (i == g.m) x = x + bc[g.right + j - 1];
    if (j == 2) x = x + bc[g.bottom + i - 1];
    if (j == g.n) x = x + bc[g.top + i - 1];
  }
  return x;
}

// ------------------------------------------------------------------------
// The passes with register ends, for plans of the fixed radices.  The
// arithmetic is that of the passes below (the same radices, twiddles and order,
// the same bits); what differs is what goes through LDS:
//  * the first stage (radix 8: M is a multiple of 4) reads its eight inputs
//    straight from the field, the second half as the odd extension's mirror
//    (its twiddles are all 1), and the last stage stores the M - 1 values that
//    are wanted straight to the field, so a transform of S stages makes S - 1
//    trips through LDS instead of S + 1;
//  * index i of a transform lies at i + i/8, which spreads the strided writes of
//    a stage over the banks (the first radix-8 stage wrote eight lanes deep
//    into one);
//  * the twiddles come from the table in memory (L1), not from a copy in LDS,
//    so a workgroup's LDS holds the two buffers only and a CU more workgroups;
//  * an index is split by a multiplication (div_by), not a division.
// What bounds them: a single field has one workgroup per tile of rows or columns
// (100 for 200 points, 512 for the columns of 1024 x 512), one or two rounds of
// the chip, and waits on a chain of a dozen barriers and loads; a batch has its
// instructions, half of them addresses, at five wavefronts per SIMD (89
// registers).  Us per field, staged -> this form, the same launch on both sides:
//   one field         rows of 200 6.8 -> 5.6, 400 7.9 -> 6.4, 1024 11.6 -> 8.2;
//                     columns of 200 10.8 -> 9.1, 400 13.3 -> 11.0, 512 (of 1023) 18.6 -> 15.3
//   batch of 8        rows of 400 2.31 -> 1.59, columns 4.31 -> 3.71
//   batch of 32       rows of 400 1.66 -> 1.19, columns 3.49 -> 2.83
//   batch of 314      rows of 200 0.43 -> 0.28, 400 1.51 -> 1.09, 512 2.59 -> 1.80;
//                     columns of 200 1.21 -> 0.58, 400 3.33 -> 2.72, 512 5.92 -> 4.51
// ------------------------------------------------------------------------
__device__ __forceinline__ int pd(int i) { return i + (i >> 3); }
__host__ __device__ inline int pd_len(int L) { return L + (L >> 3) + 1; }
// i / d by the multiplier floor(2^32 / d) + 1: exact while i d < 2^32
__device__ __forceinline__ int div_by(int i, unsigned mul) { return (int)__umulhi((unsigned)i, mul); }
__device__ __forceinline__ double2 tw_at(const double2* __restrict__ W, int byte_off) {
  return *(const double2*)((const char*)W + (unsigned)byte_off);
}

// butterfly j of a stage after the first, its inputs from a padded transform at
// ip = transform + pd(j), twiddled.  LR and Ns are multiples of 8 there (the
// first radix is 8), so pd(j + r LR) = pd(j) + r pd(LR).
template <int R>
__device__ __forceinline__ void bfly(const double2* __restrict__ ip, int pLR, int ktws,
                                     const double2* __restrict__ W, double2* v) {
  v[0] = ip[0];
  const int kb = ktws * (int)sizeof(double2);
#pragma unroll
  for (int r = 1; r < R; ++r) v[r] = cmul(ip[r * pLR], tw_at(W, r * kb));
  dft<R>(v);
}

template <int R>
__device__ __forceinline__ void stage_pd(const double2* __restrict__ in, double2* __restrict__ out, int nf,
                                         const FFTPlan& pl, int st, int Lp, int Ns) {
  const int LR = pl.L / R, tws = LR / Ns, pLR = pd(LR), pNs = pd(Ns), total = nf * LR;
  const unsigned mLR = pl.mLR[st], mNs = pl.mNs[st];
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int s = div_by(idx, mLR), j = idx - s * LR, q = div_by(j, mNs), k = j - q * Ns;
    double2 v[R];
    bfly<R>(in + s * Lp + pd(j), pLR, k * tws, pl.W, v);
    double2* op = out + s * Lp + pd(q * Ns * R + k);
#pragma unroll
    for (int r = 0; r < R; ++r) op[r * pNs] = v[r];
  }
}

// stages 1 .. nst - 2 (the first is done, the last is the caller's), with a
// barrier after each; returns the buffer that holds the result
__device__ __forceinline__ double2* mid_stages(double2* a, double2* b, int nf, const FFTPlan& pl, int Lp) {
  int Ns = 8;
  for (int st = 1; st + 1 < pl.nst; ++st) {
    const int R = pl.rad[st];
    switch (R) {
      case 8: stage_pd<8>(a, b, nf, pl, st, Lp, Ns); break;
      case 4: stage_pd<4>(a, b, nf, pl, st, Lp, Ns); break;
      case 2: stage_pd<2>(a, b, nf, pl, st, Lp, Ns); break;
      case 3: stage_pd<3>(a, b, nf, pl, st, Lp, Ns); break;
      default: stage_pd<5>(a, b, nf, pl, st, Lp, Ns); break;
    }
    __syncthreads();
    double2* t = a;
    a = b;
    b = t;
    Ns *= R;
  }
  return a;
}

// the eight inputs of first-stage butterfly j: z_t = x_t for t < M, 0 at t = 0
// and M, -x_(2M-t) above; x(t) the field's value for t = 1 .. M - 1
template <class X>
__device__ __forceinline__ void load_first(double2* v, int j, int LR, int M, X&& x) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = j + r * LR;
    const double2 p = x(t == 0 ? 1 : t), q = x(t == 0 ? 1 : M - t);
    v[r] = t == 0 ? make_double2(0.0, 0.0) : p;
    v[r + 4] = t == 0 ? make_double2(0.0, 0.0) : make_double2(-q.x, -q.y);
  }
}

// the last stage: out(s, p, value) for p = 1 .. M - 1 of every transform; the
// index runs over the transforms first where T is set (columns: adjacent
// transforms are adjacent in memory)
__device__ __forceinline__ int nf_shift(int nf) { return __ffs(nf) - 1; }
template <int R, bool T, class OUT>
__device__ __forceinline__ void last_stage_r(const double2* __restrict__ Z, int nf, const FFTPlan& pl, int Lp, OUT&& out) {
  const int LR = pl.L / R, pLR = pd(LR);
  const unsigned mLR = pl.mLR[pl.nst - 1];
  for (int idx = threadIdx.x; idx < nf * LR; idx += blockDim.x) {
    int s, k;
    if (T) {
      k = idx >> nf_shift(nf);
      s = idx & (nf - 1);
    } else {
      s = div_by(idx, mLR);
      k = idx - s * LR;
    }
    double2 v[R];
    bfly<R>(Z + s * Lp + pd(k), pLR, k, pl.W, v);
#pragma unroll
    for (int r = 0; r < (R + 1) / 2; ++r) {
      const int p = k + r * LR;
      if (p >= 1 && p < pl.M) out(s, p, v[r]);
    }
  }
}
template <bool T, class OUT>
__device__ __forceinline__ void last_stage(const double2* Z, int nf, const FFTPlan& pl, int Lp, OUT&& out) {
  switch (pl.rad[pl.nst - 1]) {
    case 8: last_stage_r<8, T>(Z, nf, pl, Lp, out); break;
    case 4: last_stage_r<4, T>(Z, nf, pl, Lp, out); break;
    case 2: last_stage_r<2, T>(Z, nf, pl, Lp, out); break;
    case 3: last_stage_r<3, T>(Z, nf, pl, Lp, out); break;
    default: last_stage_r<5, T>(Z, nf, pl, Lp, out); break;
  }
}

template <int MODE>
__device__ __forceinline__ void dst_xr_tile(const XArgs& a, int bx, int by) {
  extern __shared__ double2 sm[];
  const FFTPlan& pl = a.pl;
  const int L = pl.L, N = pl.N, rp = a.rp, Lp = pd_len(L);
  const int nrows = a.g.n - 1;
  double2* A = sm;
  double2* B = sm + rp * Lp;
  const int bsel = a.strided ? 0 : by;
  const double* __restrict__ in = a.in[bsel] ? a.in[bsel] + (long)by * a.s_in : nullptr;
  double* out = a.out[bsel] + (long)by * a.s_out;
  const double* bcb = a.bc ? a.bc + (long)by * a.s_bc : nullptr;
  const int pair0 = bx * rp;
  PointPatch pt{};
  if (MODE == X_POINTROT && !point_rows(a, pt, by, pair0, out)) return;
  const int LR = L / 8;
  for (int idx = threadIdx.x; idx < rp * LR; idx += blockDim.x) {
    const int s = div_by(idx, pl.mLR[0]), j = idx - s * LR;
    const int ra = 2 * (pair0 + s), rb = ra + 1;
    double2 v[8];
    load_first(v, j, LR, pl.M, [&](int t) {
      return make_double2(ra < nrows ? row_value<MODE>(a, pt, in, bcb, t + 1, ra + 2) : 0.0,
                          rb < nrows ? row_value<MODE>(a, pt, in, bcb, t + 1, rb + 2) : 0.0);
    });
    dft<8>(v);
#pragma unroll
    for (int r = 0; r < 8; ++r) A[s * Lp + 9 * j + r] = v[r];
  }
  __syncthreads();
  const double2* Z = mid_stages(A, B, rp, pl, Lp);
  last_stage<false>(Z, rp, pl, Lp, [&](int s, int p, double2 z) {
    const int ra = 2 * (pair0 + s), rb = ra + 1;
    const long oa = (long)ra * N + p - 1, ob = (long)rb * N + p - 1;
    if (MODE == X_SUBFROM) {
      if (ra < nrows) out[oa] = out[oa] - (-z.y);
      if (rb < nrows) out[ob] = out[ob] - z.x;
    } else {
      if (ra < nrows) out[oa] = -z.y;
      if (rb < nrows) out[ob] = z.x;
    }
  });
}

template <int MODE>
__device__ __forceinline__ void dst_yr_tile(const YArgs& a, int bx, int by) {
  extern __shared__ double2 sm[];
  const FFTPlan& pl = a.pl;
  const int L = pl.L, M = pl.M, cp = a.cp, Lp = pd_len(L);
  const int ncols = a.g.m - 1;
  const int nfft = (MODE == Y_PRED) ? 2 * cp : cp;
  double2* A = sm;
  double2* B = sm + nfft * Lp;
  const int bsel = a.strided ? 0 : by;
  const double* __restrict__ in = a.in[bsel] + (long)by * a.s_in;
  const double* __restrict__ in2 = a.in2[bsel] ? a.in2[bsel] + (long)by * a.s_in2 : nullptr;
  double* __restrict__ out = a.out[bsel] + (long)by * a.s_out;
  const int tile = (bx % 8) * a.chunk + bx / 8;  // a contiguous band of column tiles per XCD
  const int col0 = 2 * tile * cp;
  if (col0 >= ncols) return;
  const int LR = L / 8;
  for (int idx = threadIdx.x; idx < cp * LR; idx += blockDim.x) {
    const int s = idx & (cp - 1), j = idx >> nf_shift(cp);
    const int ca = col0 + 2 * s, cb = ca + 1;
    double2 v[8];
#pragma unroll
    for (int q = 0; q < (MODE == Y_PRED ? 2 : 1); ++q) {
      const double* __restrict__ f = q ? in2 : in;
      load_first(v, j, LR, M, [&](int t) {
        return make_double2(ca < ncols ? f[(long)(t - 1) * ncols + ca] : 0.0,
                            cb < ncols ? f[(long)(t - 1) * ncols + cb] : 0.0);
      });
      dft<8>(v);
#pragma unroll
      for (int r = 0; r < 8; ++r) A[(s + q * cp) * Lp + 9 * j + r] = v[r];
    }
  }
  __syncthreads();
  double2* Z = mid_stages(A, B, nfft, pl, Lp);
  if (MODE != Y_PLAIN) {
    // the spectral product, extended oddly into the other buffer
    double2* O = (Z == A) ? B : A;
    const auto put = [&](int s, int p, double ya, double yb) {
      O[s * Lp + pd(p)] = make_double2(ya, yb);
      O[s * Lp + pd(L - p)] = make_double2(-ya, -yb);
    };
    if (MODE == Y_SCALE2) {
      last_stage<true>(Z, cp, pl, Lp, [&](int s, int p, double2 z) {
        const int ca = col0 + 2 * s, cb = ca + 1;
        const double ya = (ca < ncols) ? a.tab[(long)(p - 1) * ncols + ca] * -z.y / a.div : 0.0;
        const double yb = (cb < ncols) ? a.tab[(long)(p - 1) * ncols + cb] * z.x / a.div : 0.0;
        put(s, p, ya, yb);
      });
    } else {
      // the second field's spectrum first, into the other buffer's second half
      double2* O2 = O + cp * Lp;
      last_stage<true>(Z + cp * Lp, cp, pl, Lp, [&](int s, int p, double2 z) { O2[s * Lp + pd(p)] = z; });
      __syncthreads();
      last_stage<true>(Z, cp, pl, Lp, [&](int s, int p, double2 z) {
        const int ca = col0 + 2 * s, cb = ca + 1;
        const double2 zb = O2[s * Lp + pd(p)];
        const double ba = -zb.y, bb = zb.x;
        double ya = -z.y, yb = z.x;
        // lam1i * (dst(rhs terms) + lam1 * dst(omega)), src/operators_fluid.F90:657-661
        ya = (ca < ncols) ? a.tab2[(long)(p - 1) * ncols + ca] * (ya + a.tab[(long)(p - 1) * ncols + ca] * ba) : 0.0;
        yb = (cb < ncols) ? a.tab2[(long)(p - 1) * ncols + cb] * (yb + a.tab[(long)(p - 1) * ncols + cb] * bb) : 0.0;
        put(s, p, ya, yb);
      });
    }
    for (int s = threadIdx.x; s < cp; s += blockDim.x) {
      O[s * Lp] = make_double2(0.0, 0.0);
      O[s * Lp + pd(M)] = make_double2(0.0, 0.0);
    }
    __syncthreads();
    double2* Q = (O == A) ? B : A;
    for (int idx = threadIdx.x; idx < cp * LR; idx += blockDim.x) {
      const int s = div_by(idx, pl.mLR[0]), j = idx - s * LR;
      double2 v[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = O[s * Lp + pd(j + r * LR)];
      dft<8>(v);
#pragma unroll
      for (int r = 0; r < 8; ++r) Q[s * Lp + 9 * j + r] = v[r];
    }
    __syncthreads();
    Z = mid_stages(Q, O, cp, pl, Lp);
  }
  last_stage<true>(Z, cp, pl, Lp, [&](int s, int p, double2 z) {
    const int ca = col0 + 2 * s, cb = ca + 1;
    if (ca < ncols) out[(long)(p - 1) * ncols + ca] = -z.y;
    if (cb < ncols) out[(long)(p - 1) * ncols + cb] = z.x;
  });
}

template <int MODE>
__global__ void __launch_bounds__(512) k_dst_xr(XArgs a) {
  dst_xr_tile<MODE>(a, blockIdx.x, blockIdx.y);
}
template <int MODE>
__global__ void __launch_bounds__(512) k_dst_yr(YArgs a) {
  dst_yr_tile<MODE>(a, blockIdx.x, blockIdx.y);
}

// Row pass.  Rows j0 = 0..n-2 (node j = j0+2) of length N = m-1.
template <int MODE, bool GEN>
__device__ __forceinline__ void dst_x_tile(const XArgs& a, int bx, int by) {
  extern __shared__ double2 sm[];
  const FFTPlan& pl = a.pl;
  const int L = pl.L, M = pl.M, N = pl.N, rp = a.rp;
  const int nrows = a.g.n - 1;
  double2* A = sm;
  double2* B = sm + rp * L;
  double2* Wl = sm + 2 * rp * L;
  const int bsel = a.strided ? 0 : by;
  const double* __restrict__ in = a.in[bsel] ? a.in[bsel] + (long)by * a.s_in : nullptr;
  double* out = a.out[bsel] + (long)by * a.s_out;
  const double* bcb = a.bc ? a.bc + (long)by * a.s_bc : nullptr;
  const int pair0 = bx * rp;
  PointPatch pt{};
  if (MODE == X_POINTROT && !point_rows(a, pt, by, pair0, out)) return;
  load_twiddles(Wl, pl);
  for (int idx = threadIdx.x; idx < rp * N; idx += blockDim.x) {
    const int s = idx / N;
    const int t = idx - s * N;
    const int ra = 2 * (pair0 + s), rb = ra + 1;
    const double xa = ra < nrows ? row_value<MODE>(a, pt, in, bcb, t + 2, ra + 2) : 0.0;
    const double xb = rb < nrows ? row_value<MODE>(a, pt, in, bcb, t + 2, rb + 2) : 0.0;
    A[s * L + t + 1] = make_double2(xa, xb);
    A[s * L + L - (t + 1)] = make_double2(-xa, -xb);
  }
  for (int s = threadIdx.x; s < rp; s += blockDim.x) {
    A[s * L] = make_double2(0.0, 0.0);
    A[s * L + M] = make_double2(0.0, 0.0);
  }
  __syncthreads();
  const double2* Z = fft_run<GEN>(A, B, rp, pl, Wl);
  for (int idx = threadIdx.x; idx < rp * N; idx += blockDim.x) {
    const int s = idx / N;
    const int t = idx - s * N;
    const int ra = 2 * (pair0 + s), rb = ra + 1;
    const double2 z = Z[s * L + t + 1];
    if (MODE == X_SUBFROM) {
      if (ra < nrows) out[(long)ra * N + t] = out[(long)ra * N + t] - (-z.y);
      if (rb < nrows) out[(long)rb * N + t] = out[(long)rb * N + t] - z.x;
    } else {
      if (ra < nrows) out[(long)ra * N + t] = -z.y;
      if (rb < nrows) out[(long)rb * N + t] = z.x;
    }
  }
}

// Column pass.  Columns i0 = 0..m-2 (stride m-1) of length N = n-1.
template <int MODE>
__device__ __forceinline__ void dst_y_tile(const YArgs& a, int bx, int by) {
  extern __shared__ double2 sm[];
  const FFTPlan& pl = a.pl;
  const int L = pl.L, M = pl.M, N = pl.N, cp = a.cp;
  const int ncols = a.g.m - 1;
  const int nfft = (MODE == Y_PRED) ? 2 * cp : cp;
  double2* A = sm;
  double2* B = sm + nfft * L;
  double2* Wl = sm + 2 * nfft * L;
  const int bsel = a.strided ? 0 : by;
  const double* __restrict__ in = a.in[bsel] + (long)by * a.s_in;
  const double* __restrict__ in2 = a.in2[bsel] ? a.in2[bsel] + (long)by * a.s_in2 : nullptr;
  double* __restrict__ out = a.out[bsel] + (long)by * a.s_out;
  // workgroups are dealt to the 8 XCDs round-robin: give each XCD a
  // contiguous band of column tiles so neighbouring tiles share its L2
  const int tile = (bx % 8) * a.chunk + bx / 8;
  const int col0 = 2 * tile * cp;
  if (col0 >= ncols) return;
  const int w2 = 2 * cp;  // columns handled by this workgroup
  load_twiddles(Wl, pl);
  for (int idx = threadIdx.x; idx < N * w2; idx += blockDim.x) {
    const int t = idx / w2;
    const int c = idx - t * w2;
    const int col = col0 + c;
    const int s = c >> 1;
    double v = 0.0, v2 = 0.0;
    if (col < ncols) {
      v = in[(long)t * ncols + col];
      if (MODE == Y_PRED) v2 = in2[(long)t * ncols + col];
    }
    double* pa = reinterpret_cast<double*>(&A[s * L + t + 1]);
    double* pb = reinterpret_cast<double*>(&A[s * L + L - (t + 1)]);
    pa[c & 1] = v;
    pb[c & 1] = -v;
    if (MODE == Y_PRED) {
      double* qa = reinterpret_cast<double*>(&A[(s + cp) * L + t + 1]);
      double* qb = reinterpret_cast<double*>(&A[(s + cp) * L + L - (t + 1)]);
      qa[c & 1] = v2;
      qb[c & 1] = -v2;
    }
  }
  for (int s = threadIdx.x; s < nfft; s += blockDim.x) {
    A[s * L] = make_double2(0.0, 0.0);
    A[s * L + M] = make_double2(0.0, 0.0);
  }
  __syncthreads();
  double2* Z = fft_run<true>(A, B, nfft, pl, Wl);
  if (MODE == Y_SCALE2 || MODE == Y_PRED) {
    double2* O = (Z == A) ? B : A;
    (void)O;
    for (int idx = threadIdx.x; idx < cp * N; idx += blockDim.x) {
      const int s = idx / N;
      const int t = idx - s * N;  // frequency index t+1
      const int ca = col0 + 2 * s, cb = ca + 1;
      const double2 za = Z[s * L + t + 1];
      double ya = -za.y, yb = za.x;
      if (MODE == Y_SCALE2) {
        ya = (ca < ncols) ? a.tab[(long)t * ncols + ca] * ya / a.div : 0.0;
        yb = (cb < ncols) ? a.tab[(long)t * ncols + cb] * yb / a.div : 0.0;
      } else {
        const double2 zb = Z[(s + cp) * L + t + 1];
        const double ba = -zb.y, bb = zb.x;
        // lam1i * (dst(rhs terms) + lam1 * dst(omega)), src/operators_fluid.F90:657-661
        ya = (ca < ncols) ? a.tab2[(long)t * ncols + ca] * (ya + a.tab[(long)t * ncols + ca] * ba) : 0.0;
        yb = (cb < ncols) ? a.tab2[(long)t * ncols + cb] * (yb + a.tab[(long)t * ncols + cb] * bb) : 0.0;
      }
      Z[s * L + t + 1] = make_double2(ya, yb);
      Z[s * L + L - (t + 1)] = make_double2(-ya, -yb);
    }
    for (int s = threadIdx.x; s < cp; s += blockDim.x) {
      Z[s * L] = make_double2(0.0, 0.0);
      Z[s * L + M] = make_double2(0.0, 0.0);
    }
    __syncthreads();
    double2* other = (Z == A) ? B : A;
    Z = fft_run<true>(Z, other, cp, pl, Wl);
  }
  for (int idx = threadIdx.x; idx < N * w2; idx += blockDim.x) {
    const int t = idx / w2;
    const int c = idx - t * w2;
    const int col = col0 + c;
    const int s = c >> 1;
    if (col < ncols) {
      const double2 z = Z[s * L + t + 1];
      out[(long)t * ncols + col] = (c & 1) ? z.x : -z.y;
    }
  }
}

template <int MODE, bool GEN>
__global__ void __launch_bounds__(256) k_dst_x(XArgs a) {
  dst_x_tile<MODE, GEN>(a, blockIdx.x, blockIdx.y);
}
template <int MODE>
__global__ void __launch_bounds__(256) k_dst_y(YArgs a) {
  dst_y_tile<MODE>(a, blockIdx.x, blockIdx.y);
}
template <int MODE, bool GEN>
struct DstXOp {
  using Args = XArgs;
  static __device__ __forceinline__ void tile(const XArgs& a, int bx, int by, int) { dst_x_tile<MODE, GEN>(a, bx, by); }
};
template <int MODE>
struct DstYOp {
  using Args = YArgs;
  static __device__ __forceinline__ void tile(const YArgs& a, int bx, int by, int) { dst_y_tile<MODE>(a, bx, by); }
};

// ------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------

static std::vector<int> factorize(int L) {
  std::vector<int> r;
  const int small[] = {8, 4, 2, 3, 5};
  for (int q : small)
    while (L % q == 0) {
      r.push_back(q);
      L /= q;
    }
  for (int p = 7; L > 1; p += 2)
    while (L % p == 0) {
      r.push_back(p);
      L /= p;
    }
  return r;
}

// IB_DST_FORM=fft:staged, fft:ends: see dst_tiles
static int ends_rule() {
  const char* f = std::getenv("IB_DST_FORM");
  if (f && std::strcmp(f, "fft:staged") == 0) return kEndsNever;
  if (f && std::strcmp(f, "fft:ends") == 0) return kEndsAlways;
  return 0;
}

void HostFFTPlan::init(int N) {
  dev.N = N;
  dev.M = N + 1;
  dev.L = 2 * (N + 1);
  std::vector<int> rad = factorize(dev.L);
  if ((int)rad.size() > kMaxStages) throw HipError("FFT length has too many factors");
  dev.nst = (int)rad.size();
  dev.ends = ends_rule();
  for (int i = 0, ns = 1; i < dev.nst; ns *= rad[i++]) {
    dev.rad[i] = rad[i];
    if (i >= kRegStages) continue;
    dev.mLR[i] = (unsigned)(0x100000000ull / (dev.L / rad[i])) + 1;
    dev.mNs[i] = (unsigned)(0x100000000ull / ns) + 1;
  }
  std::vector<double2> w(dev.L);
  for (int t = 0; t < dev.L; ++t) {
    long double ang = 2.0L * 3.14159265358979323846264338327950288L * (long double)t / (long double)dev.L;
    w[t] = make_double2((double)cosl(ang), (double)-sinl(ang));
  }
  IB_HIP(hipMalloc(&W, sizeof(double2) * dev.L));
  IB_HIP(hipMemcpy(W, w.data(), sizeof(double2) * dev.L, hipMemcpyHostToDevice));
  dev.W = W;
}

void HostFFTPlan::release() {
  if (W) (void)hipFree(W);
  W = nullptr;
}

size_t dst_lds_bytes(const FFTPlan& pl, int nfft) { return (size_t)(2 * nfft + 1) * pl.L * sizeof(double2); }

static size_t reg_lds_bytes(const FFTPlan& pl, int nfft) { return (size_t)2 * nfft * pd_len(pl.L) * sizeof(double2); }
// Whether a plan takes the passes with register ends: the fixed radices, from
// the lengths below on.  The form is faster at every length tried (us, one field,
// staged / register ends / matrix cores: rows of 96 points 6.1 / 5.2 / 4.6, 200
// 6.7 / 5.6 / 5.5, 256 6.6 / 5.7 / 5.7, 288 7.5 / 5.9 / 7.6, 320 7.8 / 6.3 / 7.8;
// columns of 128 9.4 / 7.7 / 9.2, 192 10.6 / 8.7 / 10.6, 200 10.7 / 9.0 / 10.9).
// The lengths are there for the results, not for speed: up to 256 points a row
// pass goes to the matrix cores, which round differently, because they beat the
// staged pass by the 10% that dst_tiles asks for; against register ends they do
// not from about 160 points on, so the field would change form and its results
// their last bits.  The lengths stand above the last such grid, which leaves the
// staged pass to rows of 260 to 319 points and to columns and strided batches
// below 200.
static bool fft_reg_plan(const FFTPlan& pl, int from) {
  return pl.ends != kEndsNever && !fft_has_generic(pl) && pl.nst >= 2 && pl.nst <= kRegStages && pl.rad[0] == 8 &&
         (pl.M >= from || pl.ends == kEndsAlways);
}
constexpr int kRegRow = 320, kRegCol = 200, kRegBatch = 200;
// a launch of tiles of `tile` pairs, nfft transforms in all (column passes
// split an index by the tile with a shift)
static bool fft_reg_ends(const FFTPlan& pl, int from, int tile, int nfft, size_t max_lds) {
  const bool ok = fft_reg_plan(pl, from) && (tile & (tile - 1)) == 0 && reg_lds_bytes(pl, nfft) <= max_lds;
  if (!ok && pl.ends == kEndsAlways)
    throw HipError("IB_DST_FORM=fft:ends: no pass with register ends for this length and tile");
  return ok;
}
// Threads: 512 from 2048 points in a workgroup's transforms on, else 256 (1.6
// points each for one transform of a field of 200, 3.1 of 400, 4 of 512 or of 1024,
// up to 16 for four pairs of predictor columns).  Us per field of a batch of 32,
// 128 / 256 / 512 threads: columns of 400 points, one pair 2.96 / 2.67 / 4.06; of
// 512 points, two pairs 10.0 / 7.9 / 7.4; rows of 400 points 1.19 / 1.09 / 1.60;
// one field's rows of 1024 points 10.4 / 8.6 / 8.1.
static int reg_threads(const FFTPlan& pl, int nfft) { return nfft * pl.L >= 2048 ? 512 : 256; }
// Pairs per workgroup of a strided batch: two up to fields of 320 points (L =
// 640), else one.  Us per field of 314 with one / two pairs: rows of 200 points
// 0.39 / 0.28, of 320 0.59 / 0.56, of 400 1.09 / 1.26, of 512 1.79 / 1.82; columns
// of 200 0.85 / 0.58, of 240 1.51 / 1.08, of 400 2.71 / 2.97, of 512 4.50 / 4.04
// (one number serves both passes).  Four pairs lose everywhere (200 points 0.34
// and 0.84).
static int reg_batch_tile(const FFTPlan& pl) { return pl.L <= 640 ? 2 : 1; }

bool fft_has_generic(const FFTPlan& pl) {
  for (int st = 0; st < pl.nst; ++st) {
    switch (pl.rad[st]) {
      case 8: case 4: case 2: case 3: case 5: break;  // the fixed radices of fft_run
      default: return true;
    }
  }
  return false;
}

namespace {
template <bool GEN>
const void* dst_x_kernel_t(int mode) {
  switch (mode) {
    case X_PLAIN: return (const void*)k_dst_x<X_PLAIN, GEN>;
    case X_APPLYBC: return (const void*)k_dst_x<X_APPLYBC, GEN>;
    case X_SUBFROM: return (const void*)k_dst_x<X_SUBFROM, GEN>;
    case X_ROT: return (const void*)k_dst_x<X_ROT, GEN>;
    case X_POINTROT: return (const void*)k_dst_x<X_POINTROT, GEN>;
    default: throw HipError("bad DST row mode");
  }
}
const void* dst_xr_kernel(int mode) {
  switch (mode) {
    case X_PLAIN: return (const void*)k_dst_xr<X_PLAIN>;
    case X_APPLYBC: return (const void*)k_dst_xr<X_APPLYBC>;
    case X_SUBFROM: return (const void*)k_dst_xr<X_SUBFROM>;
    case X_ROT: return (const void*)k_dst_xr<X_ROT>;
    case X_POINTROT: return (const void*)k_dst_xr<X_POINTROT>;
    default: throw HipError("bad DST row mode");
  }
}
const void* dst_yr_kernel(int mode) {
  switch (mode) {
    case Y_PLAIN: return (const void*)k_dst_yr<Y_PLAIN>;
    case Y_SCALE2: return (const void*)k_dst_yr<Y_SCALE2>;
    case Y_PRED: return (const void*)k_dst_yr<Y_PRED>;
    default: throw HipError("bad DST column mode");
  }
}
const void* dst_y_kernel(int mode) {
  switch (mode) {
    case Y_PLAIN: return (const void*)k_dst_y<Y_PLAIN>;
    case Y_SCALE2: return (const void*)k_dst_y<Y_SCALE2>;
    case Y_PRED: return (const void*)k_dst_y<Y_PRED>;
    default: throw HipError("bad DST column mode");
  }
}
template <bool GEN>
const void* dst_x_tab_kernel_t(int mode) {
  switch (mode) {
    case X_PLAIN: return (const void*)k_tab<DstXOp<X_PLAIN, GEN>>;
    case X_APPLYBC: return (const void*)k_tab<DstXOp<X_APPLYBC, GEN>>;
    case X_SUBFROM: return (const void*)k_tab<DstXOp<X_SUBFROM, GEN>>;
    case X_ROT: return (const void*)k_tab<DstXOp<X_ROT, GEN>>;
    default: throw HipError("DST row pass: no table kernel for this mode");
  }
}

const void* dst_x_kernel(int mode, bool gen) { return gen ? dst_x_kernel_t<true>(mode) : dst_x_kernel_t<false>(mode); }
}  // namespace

const void* dst_x_tab_kernel(int mode, bool gen) {
  return gen ? dst_x_tab_kernel_t<true>(mode) : dst_x_tab_kernel_t<false>(mode);
}
const void* dst_y_tab_kernel(int mode) {
  switch (mode) {
    case Y_SCALE2: return (const void*)k_tab<DstYOp<Y_SCALE2>>;
    case Y_PRED: return (const void*)k_tab<DstYOp<Y_PRED>>;
    default: throw HipError("DST column pass: no table kernel for this mode");
  }
}

void dst_set_max_lds(size_t bytes) {
  std::vector<const void*> fns;
  for (bool gen : {false, true}) {
    for (int mode : {X_PLAIN, X_APPLYBC, X_SUBFROM, X_ROT, X_POINTROT}) fns.push_back(dst_x_kernel(mode, gen));
    for (int mode : {X_PLAIN, X_APPLYBC, X_SUBFROM, X_ROT}) fns.push_back(dst_x_tab_kernel(mode, gen));
  }
  for (int mode : {X_PLAIN, X_APPLYBC, X_SUBFROM, X_ROT, X_POINTROT}) fns.push_back(dst_xr_kernel(mode));
  for (int mode : {Y_PLAIN, Y_SCALE2, Y_PRED}) {
    fns.push_back(dst_y_kernel(mode));
    fns.push_back(dst_yr_kernel(mode));
  }
  for (int mode : {Y_SCALE2, Y_PRED}) fns.push_back(dst_y_tab_kernel(mode));
  for (const void* f : fns) IB_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

TabEntry<XArgs> dst_x_entry(const FFTPlan& pl, const DstLaunch& l, const Geom& g, int rp, size_t max_lds,
                            size_t* lds) {
  TabEntry<XArgs> e{};
  XArgs& a = e.a;
  const bool strided = l.strided;
  if (!strided && l.batch > kMaxBatch) throw HipError("DST row pass: batch > 4 needs strides");
  if (!strided && (l.s_in || l.s_out || l.s_bc)) throw HipError("DST row pass: strides on an unstrided batch");
  a.strided = strided;
  for (int b = 0; b < (strided ? 1 : l.batch); ++b) {
    a.in[b] = l.in[b];
    a.out[b] = l.out[b];
  }
  a.s_in = l.s_in;
  a.s_out = l.s_out;
  a.s_bc = l.s_bc;
  a.c0 = l.c0;
  a.w = l.w;
  a.key = l.key;
  a.bc = l.bc;
  a.hx = l.hx;
  a.hy = l.hy;
  a.g = g;
  a.pl = pl;
  while (rp > 1 && dst_lds_bytes(pl, rp) > max_lds) rp /= 2;
  a.rp = rp;
  const int npairs = ceil_div(g.n - 1, 2);
  e.nbx = ceil_div(npairs, rp);
  e.nby = l.batch;
  *lds = dst_lds_bytes(pl, rp);
  if (*lds > max_lds) throw HipError("DST row pass needs more LDS than the device allows");
  return e;
}

TabEntry<YArgs> dst_y_entry(const FFTPlan& pl, int mode, const DstLaunch& l, const Geom& g, int cp,
                            size_t max_lds, size_t* lds) {
  TabEntry<YArgs> e{};
  YArgs& a = e.a;
  const bool strided = l.strided;
  if (!strided && l.batch > kMaxBatch) throw HipError("DST column pass: batch > 4 needs strides");
  if (!strided && (l.s_in || l.s_in2 || l.s_out)) throw HipError("DST column pass: strides on an unstrided batch");
  a.strided = strided;
  for (int b = 0; b < (strided ? 1 : l.batch); ++b) {
    a.in[b] = l.in[b];
    a.in2[b] = l.in2[b];
    a.out[b] = l.out[b];
  }
  a.s_in = l.s_in;
  a.s_in2 = l.s_in2;
  a.s_out = l.s_out;
  a.tab = l.tab;
  a.tab2 = l.tab2;
  a.div = l.div;
  a.g = g;
  a.pl = pl;
  const int mult = (mode == Y_PRED) ? 2 : 1;
  while (cp > 1 && dst_lds_bytes(pl, mult * cp) > max_lds) cp /= 2;
  a.cp = cp;
  const int npairs = ceil_div(g.m - 1, 2);
  const int ntiles = ceil_div(npairs, cp);
  a.chunk = ceil_div(ntiles, 8);
  e.nbx = 8 * a.chunk;
  e.nby = l.batch;
  *lds = dst_lds_bytes(pl, mult * cp);
  if (*lds > max_lds) throw HipError("DST column pass needs more LDS than the device allows");
  return e;
}

void dst_x(hipStream_t st, const FFTPlan& pl, int mode, const DstLaunch& l, const Geom& g, int rp,
           size_t max_lds) {
  size_t lds = 0;
  const TabEntry<XArgs> e = dst_x_entry(pl, l, g, rp, max_lds, &lds);
  void* args[] = {(void*)&e.a};
  if (fft_reg_ends(pl, l.strided ? kRegBatch : kRegRow, e.a.rp, e.a.rp, max_lds))
    IB_HIP(hipLaunchKernel(dst_xr_kernel(mode), dim3(e.nbx, e.nby), dim3(reg_threads(pl, e.a.rp)), args,
                           reg_lds_bytes(pl, e.a.rp), st));
  else
    IB_HIP(hipLaunchKernel(dst_x_kernel(mode, fft_has_generic(pl)), dim3(e.nbx, e.nby), dim3(256), args, lds, st));
  IB_LAUNCH_CHECK();
}

void dst_y(hipStream_t st, const FFTPlan& pl, int mode, const DstLaunch& l, const Geom& g, int cp,
           size_t max_lds) {
  size_t lds = 0;
  const TabEntry<YArgs> e = dst_y_entry(pl, mode, l, g, cp, max_lds, &lds);
  void* args[] = {(void*)&e.a};
  const int nfft = (mode == Y_PRED ? 2 : 1) * e.a.cp;
  if (fft_reg_ends(pl, l.strided ? kRegBatch : kRegCol, e.a.cp, nfft, max_lds))
    IB_HIP(hipLaunchKernel(dst_yr_kernel(mode), dim3(e.nbx, e.nby), dim3(reg_threads(pl, nfft)), args,
                           reg_lds_bytes(pl, nfft), st));
  else
    IB_HIP(hipLaunchKernel(dst_y_kernel(mode), dim3(e.nbx, e.nby), dim3(256), args, lds, st));
  IB_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------
// Form and tile shapes of the DST passes, picked by timing.  The row pairs
// per workgroup of the row pass (rp) and the column pairs of the column pass
// (cp) decide only how many transforms share a workgroup's LDS, never a
// transform's arithmetic, so every choice gives the same bits.  The
// matrix-core form (ib_dst_dense.hip) sums in another order: it is taken for
// a pass class only when it is at least 10% faster, so that a near tie does
// not flip between processes.  Each candidate that fits runs a few times on
// scratch fields between HIP events; the fastest is kept for the process,
// per grid shape.  Two classes are timed: one field per launch (the time
// step) and a strided batch of 8 fields (the Schur assembly, whose launches
// cover hundreds of columns).  The Stockham tiles are timed for one field; the
// batch takes the same ones, or reg_batch_tile's for the passes with register
// ends.
//
// IB_DST_TILES=rp,cp forces the Stockham tiles; IB_DST_TUNE=0 keeps the
// fixed rule (rp 2 up to transform length 512, else 1; cp 1); neither times
// anything.  IB_DST_FORM=fft keeps the Stockham form (=fft:staged without
// register ends, =fft:ends with them at every length: an error where a pass
// has none; tests compare the two), =dense takes the
// matrix-core form for both classes (its fastest configuration, or the
// (T, KS) = (1, 8) configuration when nothing is timed), =dense:k the matrix-core
// form in configuration k without timing, =auto (the default) times.
namespace {
std::mutex g_tile_mu;
std::map<std::array<long, 6>, DstTiles> g_tiles;
constexpr int kDenseDefault = 1;
constexpr int kTuneBatch = 8;

template <class F>
float time_launches(hipStream_t st, F&& launch) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  IB_HIP(hipEventCreate(&e0));
  IB_HIP(hipEventCreate(&e1));
  float best = 1e30f;
  try {
    launch();  // warm-up (code objects, caches)
    launch();
    for (int rep = 0; rep < 3; ++rep) {
      IB_HIP(hipEventRecord(e0, st));
      for (int k = 0; k < 4; ++k) launch();
      IB_HIP(hipEventRecord(e1, st));
      IB_HIP(hipEventSynchronize(e1));
      float ms = 0.0f;
      IB_HIP(hipEventElapsedTime(&ms, e0, e1));
      best = std::min(best, ms);
    }
  } catch (...) {
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    throw;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return best / 4.0f;
}

// 0 auto, 1 Stockham only, 2 matrix-core form, 3 matrix-core form in
// configuration *cfg
int form_rule(int* cfg) {
  const char* f = std::getenv("IB_DST_FORM");
  if (!f || !*f || std::strcmp(f, "auto") == 0) return 0;
  if (std::strcmp(f, "fft") == 0 || ends_rule() != 0) return 1;
  if (std::strcmp(f, "dense") == 0) return 2;
  int k = -1;
  char tail = 0;
  if (std::sscanf(f, "dense:%d%c", &k, &tail) == 1 && k >= 0 && k < kDenseCfgs) {
    *cfg = k;
    return 3;
  }
  throw HipError("IB_DST_FORM must be fft, fft:staged, fft:ends, dense, dense:k (0 <= k < 5) or auto");
}

struct Scratch {
  double* p = nullptr;
  ~Scratch() {
    if (p) (void)hipFree(p);
  }
};
}  // namespace

DstTiles dst_tiles(hipStream_t st, const FFTPlan& px, const FFTPlan& py, const DenseMat* dx, const DenseMat* dy,
                   double* tq, const Geom& g, size_t max_lds) {
  DstTiles t;
  t.rp = px.L <= 512 ? 2 : 1;
  t.cp = 1;
  t.rp_b = t.rp;
  int forced_cfg = kDenseDefault;
  const int rule = form_rule(&forced_cfg);
  const bool dense_ok = dx && dy && dx->S && dy->S && tq;
  if (rule >= 2 && !dense_ok) throw HipError("IB_DST_FORM=dense: no sine matrices");
  const int fixed_form = rule >= 2 ? forced_cfg + 1 : 0;
  if (const char* f = std::getenv("IB_DST_TILES")) {
    int rp = 0, cp = 0;
    if (std::sscanf(f, "%d,%d", &rp, &cp) != 2 || rp < 1 || rp > 8 || cp < 1 || cp > 8)
      throw HipError("IB_DST_TILES must be rp,cp with 1 <= rp, cp <= 8");
    t.rp = rp;  // dst_x_entry / dst_y_entry halve a choice the LDS cannot hold
    t.cp = cp;
    t.rp_b = rp;
    t.cp_b = cp;
    t.xform = t.yform = t.xform_b = t.yform_b = fixed_form;
    t.source = 2;
    return t;
  }
  if (const char* f = std::getenv("IB_DST_TUNE"))
    if (std::strcmp(f, "0") == 0) {
      t.xform = t.yform = t.xform_b = t.yform_b = fixed_form;
      return t;
    }
  if (rule == 3) {  // a forced configuration: the Stockham tiles keep the fixed rule
    t.xform = t.yform = t.xform_b = t.yform_b = fixed_form;
    t.source = 2;
    return t;
  }
  const bool try_dense = dense_ok && rule != 1;
  const std::array<long, 6> key{g.m, g.n, px.L, py.L, (long)max_lds, (long)(px.ends * 8 + rule * 2 + (try_dense ? 1 : 0))};
  std::lock_guard<std::mutex> lock(g_tile_mu);
  auto it = g_tiles.find(key);
  if (it != g_tiles.end()) return it->second;
  const long P = g.P;
  Scratch in, out;
  const size_t bytes = sizeof(double) * (size_t)P * kTuneBatch;
  IB_HIP(hipMalloc(&in.p, bytes));
  IB_HIP(hipMalloc(&out.p, bytes));
  IB_HIP(hipMemsetAsync(in.p, 0, bytes, st));
  // one field per launch: the Stockham tiles, then the matrix-core configurations
  DstLaunch lx;
  lx.in[0] = in.p;
  lx.out[0] = out.p;
  DstLaunch ly = lx;
  ly.tab = in.p;  // any table: the values do not change the time
  ly.div = 1.0;
  float best = 1e30f;
  for (int rp : {1, 2, 4}) {
    if (dst_lds_bytes(px, rp) > max_lds) continue;
    const float ms = time_launches(st, [&] { dst_x(st, px, X_PLAIN, lx, g, rp, max_lds); });
    if (ms < best) {
      best = ms;
      t.rp = rp;
    }
  }
  t.us[0] = best * 1e3f;
  best = 1e30f;
  for (int cp : {1, 2, 4}) {
    if (dst_lds_bytes(py, cp) > max_lds) continue;
    const float ms = time_launches(st, [&] { dst_y(st, py, Y_SCALE2, ly, g, cp, max_lds); });
    if (ms < best) {
      best = ms;
      t.cp = cp;
    }
  }
  t.us[2] = best * 1e3f;
  // a strided batch of kTuneBatch fields
  DstLaunch bx = lx;
  bx.batch = kTuneBatch;
  bx.strided = true;
  bx.s_in = bx.s_out = P;
  DstLaunch by = bx;
  by.tab = in.p;
  by.div = 1.0;
  t.rp_b = fft_reg_plan(px, kRegBatch) ? reg_batch_tile(px) : t.rp;
  t.cp_b = fft_reg_plan(py, kRegBatch) ? reg_batch_tile(py) : t.cp;
  t.us[4] = time_launches(st, [&] { dst_x(st, px, X_PLAIN, bx, g, t.rp_b, max_lds); }) * 1e3f / kTuneBatch;
  t.us[6] = time_launches(st, [&] { dst_y(st, py, Y_SCALE2, by, g, t.cp_b, max_lds); }) * 1e3f / kTuneBatch;
  if (try_dense) {
    // a class is timed only if the matrix-core form could beat the measured
    // Stockham time at the FP64 matrix peak (78.6 TFLOP/s; 2N flops per
    // point and product, two products in the column pass); IB_DST_FORM=dense
    // times every class
    const double peak = 78.6e6;  // flop per microsecond
    const double lb[4] = {2.0 * (g.m - 1) * P / peak, 4.0 * (g.n - 1) * P / peak,
                          2.0 * (g.m - 1) * P / peak, 4.0 * (g.n - 1) * P / peak};
    float best_us[4] = {1e30f, 1e30f, 1e30f, 1e30f};
    int cfg[4] = {kDenseDefault, kDenseDefault, kDenseDefault, kDenseDefault};
    const DstLaunch* ls[4] = {&lx, &ly, &bx, &by};
    for (int q = 0; q < 4; ++q) {
      const float fft_us = t.us[2 * q];
      if (rule != 2 && lb[q] >= fft_us) continue;
      const int nf = q < 2 ? 1 : kTuneBatch;
      for (int c = 0; c < kDenseCfgs; ++c) {
        const float us = 1e3f / nf * time_launches(st, [&] {
          if (q % 2 == 0) dst_dense_x(st, *dx, X_PLAIN, *ls[q], g, c);
          else dst_dense_y(st, *dy, Y_SCALE2, *ls[q], g, c, tq, kMaxBatch);
        });
        if (us < best_us[q]) {
          best_us[q] = us;
          cfg[q] = c;
        }
      }
      t.us[2 * q + 1] = best_us[q];
    }
    const auto pick = [&](int q) {
      if (rule == 2) return cfg[q] + 1;
      return (t.us[2 * q + 1] >= 0.0f && t.us[2 * q + 1] < 0.9f * t.us[2 * q]) ? cfg[q] + 1 : 0;
    };
    t.xform = pick(0);
    t.yform = pick(1);
    t.xform_b = pick(2);
    t.yform_b = pick(3);
  }
  IB_HIP(hipStreamSynchronize(st));
  t.source = 1;
  g_tiles[key] = t;
  return t;
}

}  // namespace ibg
