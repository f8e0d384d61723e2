// ib_gmres.hip -- device-resident restarted GMRES for the FSI Schur system.
//
// Follows PETSc 3.11 KSPGMRES as configured by setup_ksp
// (src/variables.F90:565-574): no preconditioner, unpreconditioned residual
// norm, nonzero initial guess, classical Gram-Schmidt without refinement,
// Givens-rotation residual estimate, convergence when
// ||r|| <= max(rtol*||b||, atol), divergence when ||r|| >= 1e4*||b||, happy
// breakdown tolerance 1e-30.  The Krylov basis, Hessenberg matrix and
// rotations stay in HBM; the host reads the small status block only.
//
// Every kernel returns at once when the status block already carries a
// convergence reason, so the host may enqueue several iterations ahead of
// the status it has read (the extra matvecs then write only into basis
// columns the solution never uses).
#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <vector>

#include "ib_device.h"
#include "ib_kernels.h"

namespace ibg {

constexpr int kGmT = 1024;

__device__ double gm_block_sum(double v, double* sh) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (t < s) sh[t] = sh[t] + sh[t + s];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = warpSize / 2; o > 0; o >>= 1) v += __shfl_down(v, o);
  return v;
}

// V0 = b - A x; residual norm, initial tolerance and convergence tests
__global__ void __launch_bounds__(kGmT) k_gm_start(int nf, const double* __restrict__ b, const double* __restrict__ Ax,
                                                   double* __restrict__ V, GmresDev* s, double* grs, double rtol,
                                                   double atol) {
  __shared__ double sh[kGmT];
  double pr = 0.0, pb = 0.0;
  for (int i = threadIdx.x; i < nf; i += blockDim.x) {
    const double r = b[i] - Ax[i];
    V[i] = r;
    pr += r * r;
    pb += b[i] * b[i];
  }
  const double res = sqrt(gm_block_sum(pr, sh));
  const double bn = sqrt(gm_block_sum(pb, sh));
  __shared__ int s_reason;
  if (threadIdx.x == 0) {
    if (s->first) {
      s->bnorm = bn;
      s->rn0 = bn > 0.0 ? bn : res;
      s->ttol = fmax(rtol * s->rn0, atol);
      s->first = 0;
    }
    grs[0] = res;
    s->res = res;
    s->it = 0;
    int reason = 0;
    if (res == 0.0 || res <= s->ttol) reason = 1;
    else if (res >= 1e4 * s->rn0) reason = -1;
    s->reason = reason;
    s_reason = reason;
  }
  __syncthreads();
  if (s_reason == 0) {
    const double inv = res;
    for (int i = threadIdx.x; i < nf; i += blockDim.x) V[i] = V[i] / inv;
  }
}

// h_j = <w, v_j> for j = 0..it, w = V[it+1] unmodified (classical
// Gram-Schmidt); one wavefront per dot product, many workgroups.
__global__ void __launch_bounds__(256) k_gm_dots(int nf, int kmax, const double* __restrict__ V,
                                                 const GmresDev* __restrict__ s, double* __restrict__ H) {
  if (s->reason) return;
  const int it = s->it;
  const int j = (blockIdx.x * blockDim.x + threadIdx.x) / warpSize;
  const int lane = threadIdx.x % warpSize;
  if (j > it) return;
  const double* w = V + (long)(it + 1) * nf;
  const double* vj = V + (long)j * nf;
  double p = 0.0;
  for (int i = lane; i < nf; i += warpSize) p += w[i] * vj[i];
  p = wave_sum(p);
  if (lane == 0) H[(long)it * (kmax + 1) + j] = p;
}

// KSPGMRESBuildSoln: back substitution on the rotated Hessenberg, x += V y.
// Columns of H are staged in LDS in chunks of `bs` columns so the dependent
// chain of the substitution runs on LDS values.
static int bs_chunk(int kmax) {
  int c = 6000 / (kmax + 1) - 2;  // keep (c + 2)(kmax + 1) doubles under 48 KB
  return c > 16 ? 16 : (c < 1 ? 1 : c);
}

__global__ void __launch_bounds__(kGmT) k_gm_buildsol(int nf, int kmax, int kBsChunk, const double* __restrict__ V,
                                                      GmresDev* s, const double* __restrict__ H,
                                                      const double* __restrict__ grs, double* __restrict__ x,
                                                      double* __restrict__ nrs) {
  extern __shared__ double dyn[];  // t[kmax+1] | y[kmax+1] | chunk[kBsChunk][kmax+1]
  const int it = s->it;  // number of Arnoldi vectors used
  if (it <= 0) return;
  const int ld = kmax + 1;
  double* t = dyn;
  double* y = dyn + ld;
  double* chunk = dyn + 2 * ld;
  const int top = it - 1;
  for (int j = threadIdx.x; j <= top; j += blockDim.x) t[j] = grs[j];
  __syncthreads();
  for (int k1 = top; k1 >= 0; k1 -= kBsChunk) {
    const int k0 = k1 - kBsChunk + 1 < 0 ? 0 : k1 - kBsChunk + 1;
    const int nc = k1 - k0 + 1;
    // stage columns k0..k1, rows 0..k1
    for (int q = threadIdx.x; q < nc * (k1 + 1); q += blockDim.x) {
      const int c = q / (k1 + 1), r = q - c * (k1 + 1);
      chunk[c * ld + r] = H[(long)(k0 + c) * ld + r];
    }
    __syncthreads();
    for (int k = k1; k >= k0; --k) {
      const double* col = chunk + (k - k0) * ld;
      if (threadIdx.x == 0) y[k] = t[k] / col[k];
      __syncthreads();
      const double yk = y[k];
      for (int j = threadIdx.x; j < k; j += blockDim.x) t[j] = t[j] - col[j] * yk;
      __syncthreads();
    }
  }
  for (int j = threadIdx.x; j <= top; j += blockDim.x) nrs[j] = y[j];
  for (int i = threadIdx.x; i < nf; i += blockDim.x) {
    double acc = 0.0;
    for (int j = 0; j <= top; ++j) acc += y[j] * V[(long)j * nf + i];
    x[i] = x[i] + acc;
  }
}

// y = S x, S dense nf x nf column major.  A workgroup owns 16 rows and
// splits the columns into 16 contiguous groups (4 per wavefront: lane & 15
// is the row, lane >> 4 the group), so the matrix streams through many CUs;
// the 16 partial sums of a row are added in group order.
struct GemvOp {
  using Args = GemvArgs;
  static __device__ __forceinline__ void tile(const GemvArgs& a, int bx, int by, int);
};

__device__ __forceinline__ void GemvOp::tile(const GemvArgs& a, int bx, int, int) {
  __shared__ double part[16][16];
  const int nf = a.nf;
  const double* __restrict__ S = a.S;
  const double* __restrict__ x = a.x;
  double* __restrict__ y = a.y;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rl = lane & 15, grp = wv * 4 + (lane >> 4);
  const int r = bx * 16 + rl;
  const int per = (nf + 15) / 16;
  const int j0 = min(nf, grp * per), j1 = min(nf, j0 + per);
  double acc = 0.0;
  if (r < nf) {
    for (int j = j0; j < j1; j += 8) {
      double sv[8], xv[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int jj = min(j + c, j1 - 1);
        sv[c] = S[(long)jj * nf + r];
        xv[c] = x[jj];
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) acc += (j + c < j1 ? sv[c] : 0.0) * xv[c];
    }
  }
  part[grp][rl] = acc;
  __syncthreads();
  if (threadIdx.x < 16 && r < nf) {
    double a = part[0][rl];
    for (int q = 1; q < 16; ++q) a += part[q][rl];
    y[r] = a;
  }
}

__global__ void __launch_bounds__(256) k_gemv(GemvArgs a) { GemvOp::tile(a, blockIdx.x, 0, 0); }

TabEntry<GemvArgs> gemv_entry(int nf, const double* S, const double* x, double* y) {
  TabEntry<GemvArgs> e{};
  e.a = GemvArgs{nf, S, x, y};
  e.nbx = ceil_div(std::max(nf, 1), 16);
  e.nby = 1;
  return e;
}

const void* gemv_tab_kernel() { return (const void*)k_tab<GemvOp>; }

void gemv(hipStream_t st, int nf, const double* S, const double* x, double* y) {
  if (nf <= 0) return;
  const TabEntry<GemvArgs> e = gemv_entry(nf, S, x, y);
  hipLaunchKernelGGL(k_gemv, dim3(e.nbx), dim3(256), 0, st, e.a);
  IB_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------
// Whole solve in one workgroup for a dense Schur matrix.  The same PETSc
// 3.11 GMRES as the kernels above (CGS, Givens, restart, stopping tests),
// but every iteration stays inside the kernel: S is held in registers
// (MAXC columns of one row per thread, the rest read from L2), w, the new
// Hessenberg column, the rotations and the residual vector in LDS, and the
// Krylov basis in HBM/L2.  Iterations cost a few microseconds instead of
// three dependent launches.
// ------------------------------------------------------------------------
struct GmDenseArgs {
  int nf, kmax, maxit;
  int nvl;     // basis vectors held in LDS (the rest are read from HBM/L2)
  int bsc;     // Hessenberg columns staged per back-substitution chunk
  const double* S;
  const double* b;
  double* x;
  double* V;
  double* H;
  GmresDev* s;
  double rtol, atol;
};

constexpr int kGmRem = 12;  // S entries per thread fetched from L2 in one unrolled batch

// acc += -sum_{j in [q0, q1)} h[j] * v_j[r] in j order, v_j from the LDS cache
// for j < nvl and from HBM/L2 otherwise; loads are issued in batches of 8.
__device__ __forceinline__ double gm_axpy_col(double acc, const double* __restrict__ h, const double* cache,
                                              const double* __restrict__ V, int nf, int nvl, int q0, int q1,
                                              int r) {
  const int qa = min(q1, nvl);
  for (int j = q0; j < qa; j += 8) {
    double v[8], hv[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int jj = min(j + c, qa - 1);
      v[c] = cache[(long)jj * nf + r];
      hv[c] = h[jj];
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) acc += -(j + c < qa ? hv[c] : 0.0) * v[c];
  }
  for (int j = max(q0, nvl); j < q1; j += 8) {
    double v[8], hv[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int jj = min(j + c, q1 - 1);
      v[c] = V[(long)jj * nf + r];
      hv[c] = h[jj];
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) acc += -(j + c < q1 ? hv[c] : 0.0) * v[c];
  }
  return acc;
}

// The thread index as a value the compiler cannot see through: per-thread
// addresses derived from it are recomputed in each phase instead of being
// hoisted out of the solve loop and kept live in registers for the whole
// kernel (which would crowd out the register-resident part of S).
__device__ __forceinline__ int gm_opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Cross-lane data movement through DPP (register-level, no LDS crossbar).
// CTRL is the gfx9 dpp_ctrl code; doubles move as two 32-bit halves.
template <int CTRL>
__device__ __forceinline__ double gm_dpp(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// every lane gets the sum over its row of 16 lanes: quad_perm [1,0,3,2],
// quad_perm [2,3,0,1], row_ror:4, row_ror:8
__device__ __forceinline__ double gm_row_sum16(double v) {
  v += gm_dpp<0xB1>(v);
  v += gm_dpp<0x4E>(v);
  v += gm_dpp<0x124>(v);
  v += gm_dpp<0x128>(v);
  return v;
}

__device__ __forceinline__ double gm_readlane(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sum over the 64 lanes of a wavefront (uniform result, fixed order)
__device__ __forceinline__ double gm_wave_sum(double v) {
  const double rs = gm_row_sum16(v);
  return (gm_readlane(rs, 0) + gm_readlane(rs, 16)) + (gm_readlane(rs, 32) + gm_readlane(rs, 48));
}

// sum over i = sub, sub+16, ... < nf of w[i] v[i], in batches of 8 loads
// per operand with clamped indices (no branches between the loads)
template <bool LDS>
__device__ __forceinline__ double gm_dot16(const double* w, const double* v, int nf, int sub) {
  double p = 0.0;
  for (int i0 = sub; i0 < nf; i0 += 16 * 8) {
    double wv[8], vv[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int i = min(i0 + 16 * c, nf - 1);
      wv[c] = w[i];
      vv[c] = v[i];
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) p += (i0 + 16 * c < nf ? wv[c] : 0.0) * vv[c];
  }
  return p;
}

template <int CTRL, int RM>
__device__ __forceinline__ double gm_dpp_old(double v, double old) {
  const long long b = __double_as_longlong(v), o = __double_as_longlong(old);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, CTRL, RM, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), CTRL, RM, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <int CTRL, int RM>
__device__ __forceinline__ void gm_scan_step(double& A, double& B) {
  const double Ap = gm_dpp_old<CTRL, RM>(A, 1.0), Bp = gm_dpp_old<CTRL, RM>(B, 0.0);
  B = A * Bp + B;
  A = A * Ap;
}
// inclusive scan of the affine maps x -> A x + B over the 64 lanes (lane l
// ends with f_l o ... o f_0): row_shr 1/2/4/8 within rows of 16, then
// row_bcast 15 and 31 across rows; lanes a shift leaves without a source
// compose with the identity (1, 0)
__device__ __forceinline__ void gm_affine_scan(double& A, double& B) {
  gm_scan_step<0x111, 0xF>(A, B);
  gm_scan_step<0x112, 0xF>(A, B);
  gm_scan_step<0x114, 0xF>(A, B);
  gm_scan_step<0x118, 0xF>(A, B);
  gm_scan_step<0x142, 0xA>(A, B);
  gm_scan_step<0x143, 0xC>(A, B);
}
// the value of lane l-1 (wave_shr 1); lane 0 gets `first`
__device__ __forceinline__ double gm_shift_up1(double v, double first) { return gm_dpp_old<0x138, 0xF>(v, first); }

// row-segment layout of the matrix-vector product: thread (seg, r) owns row
// r and columns [j0, j1); nseg segments of nf threads
struct GmLayout {
  int nseg, seg, r, j0, j1;
  bool act;
  __device__ GmLayout(int t, int nf, int T) {
    nseg = nf <= T ? min(16, T / nf) : 1;
    seg = t / nf;
    r = t - seg * nf;
    act = nf <= T && seg < nseg;
    const int per = (nf + nseg - 1) / nseg;
    j0 = act ? seg * per : 0;
    j1 = act ? min(nf, j0 + per) : 0;
  }
};

// part[0*nf+i] + part[1*nf+i] + ... + part[(nseg-1)*nf+i] in that order (nseg <= 16)
__device__ __forceinline__ double gm_sum_parts(const double* part, int nf, int i, int nseg) {
  double v[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) v[q] = part[min(q, nseg - 1) * nf + i];
  double acc = v[0];
#pragma unroll
  for (int q = 1; q < 16; ++q) acc += (q < nseg ? v[q] : 0.0);
  return acc;
}

__device__ __forceinline__ double gm_block_sum2(double v, double* red, int T) {
  const int t = gm_opaque(threadIdx.x);
  v = gm_wave_sum(v);
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  double tot = 0.0;
  for (int q = 0; q < T / 64; ++q) tot += red[q];
  __syncthreads();
  return tot;
}

// out = S vin (vin, out in LDS); S entries [j0, j0+MAXC) of the thread's row
// segment come from registers, the rest from L2 in unrolled batches.  Ends
// with a barrier.
template <int MAXC>
__device__ __forceinline__ void gm_gemv(const double (&sreg)[MAXC], const double* __restrict__ S, int nf, int T,
                                        const double* vin, double* out, double* part) {
  const GmLayout g(gm_opaque(threadIdx.x), nf, T);
  if (nf <= T) {
    // branch-free (clamped indices, zero weights past the segment) so that
    // all loads of a batch are in flight together
    if (g.act) {
      double acc = 0.0;
#pragma unroll
      for (int c0 = 0; c0 < MAXC; c0 += 8) {
        double vv[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) vv[c] = c0 + c < MAXC ? vin[min(g.j0 + c0 + c, nf - 1)] : 0.0;
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (c0 + c < MAXC) acc += sreg[c0 + c] * vv[c];  // sreg is 0 past the segment
      }
      for (int jb = g.j0 + MAXC; jb < g.j1; jb += kGmRem) {
        double sv[kGmRem], xv[kGmRem];
#pragma unroll
        for (int c = 0; c < kGmRem; ++c) {
          const int j = min(jb + c, g.j1 - 1);
          sv[c] = S[(long)j * nf + g.r];
          xv[c] = vin[j];
        }
#pragma unroll
        for (int c = 0; c < kGmRem; ++c) acc += (jb + c < g.j1 ? sv[c] : 0.0) * xv[c];
      }
      part[g.seg * nf + g.r] = acc;
    }
    __syncthreads();
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) out[i] = gm_sum_parts(part, nf, i, g.nseg);
  } else {
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
      double acc = 0.0;
      for (int j = 0; j < nf; ++j) acc += S[(long)j * nf + i] * vin[j];
      out[i] = acc;
    }
  }
  __syncthreads();
}

template <int MAXC>
__global__ void __launch_bounds__(kGmT) k_gmres_dense(GmDenseArgs a) {
  extern __shared__ double dyn[];
  const int nf = a.nf, kmax = a.kmax, ld = kmax + 1, T = kGmT;
  double* vl = dyn;               // nf: the basis vector being multiplied
  double* wl = vl + nf;           // nf: w
  double* hcol = wl + nf;         // kmax + 2
  double* lcc = hcol + kmax + 2;  // kmax
  double* lss = lcc + kmax;       // kmax
  double* grs = lss + kmax;       // kmax + 1
  double* yv = grs + kmax + 1;    // kmax + 1
  double* part = yv + kmax + 1;   // T
  double* cache = part + T;       // basis vectors 0..nvl-1; Hessenberg chunks in the back substitution
  const int nvl = a.nvl;
  __shared__ double red[kGmT / 64];
  __shared__ double s_val[2];
  __shared__ int s_flag[2];

  double sreg[MAXC];  // the first MAXC columns of the thread's row segment, for the whole solve
  {
    const GmLayout g(threadIdx.x, nf, T);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) sreg[c] = (g.j0 + c < g.j1) ? a.S[(long)(g.j0 + c) * nf + g.r] : 0.0;
  }

  int its = 0, reason = 0, first = 1;
  double rn0 = 0.0, ttol = 0.0;
  while (true) {
    // ---- cycle start: r = b - S x
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) vl[i] = a.x[i];
    __syncthreads();
    gm_gemv<MAXC>(sreg, a.S, nf, T, vl, wl, part);
    double pr = 0.0, pb = 0.0;
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
      const double rv = a.b[i] - wl[i];
      wl[i] = rv;
      pr += rv * rv;
      pb += a.b[i] * a.b[i];
    }
    const double res0 = sqrt(gm_block_sum2(pr, red, T));
    const double bn = sqrt(gm_block_sum2(pb, red, T));
    if (first) {
      rn0 = bn > 0.0 ? bn : res0;
      ttol = fmax(a.rtol * rn0, a.atol);
      first = 0;
    }
    if (res0 == 0.0 || res0 <= ttol) reason = 1;
    else if (res0 >= 1e4 * rn0) reason = -1;
    if (reason) break;
    if (threadIdx.x == 0) grs[0] = res0;
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
      const double v0 = wl[i] / res0;
      vl[i] = v0;
      a.V[i] = v0;
      if (nvl > 0) cache[i] = v0;
    }
    __syncthreads();
    int it = 0;
    while (true) {
      gm_gemv<MAXC>(sreg, a.S, nf, T, vl, wl, part);  // w = S v_it
      // classical Gram-Schmidt coefficients h_j = <w, v_j>, j = 0..it: one
      // row of 16 lanes per coefficient, reduced with DPP
      {
        const int t = gm_opaque(threadIdx.x);
        const int sub = t & 15;
        const int ndots = it + 1;
        for (int j = t >> 4; j < ndots; j += T / 16) {
          double p = 0.0;
          if (j < nvl) p = gm_dot16<true>(wl, cache + (long)j * nf, nf, sub);
          else p = gm_dot16<false>(wl, a.V + (long)j * nf, nf, sub);
          p = gm_row_sum16(p);
          if (sub == 0) hcol[j] = p;
        }
      }
      __syncthreads();
      // w -= sum_j h_j v_j (j range split over the row segments, partials in fixed order), ||w||
      double pn = 0.0;
      {
        const GmLayout g(gm_opaque(threadIdx.x), nf, T);
        const int jn = it + 1;
        if (nf <= T && g.nseg > 1) {
          const int per2 = (jn + g.nseg - 1) / g.nseg;
          if (g.act) {
            const int q0 = min(jn, g.seg * per2), q1 = min(jn, q0 + per2);
            part[g.seg * nf + g.r] = gm_axpy_col(0.0, hcol, cache, a.V, nf, nvl, q0, q1, g.r);
          }
          __syncthreads();
          for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
            const double acc = wl[i] + gm_sum_parts(part, nf, i, g.nseg);
            wl[i] = acc;
            pn += acc * acc;
          }
        } else {
          for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
            const double acc = gm_axpy_col(wl[i], hcol, cache, a.V, nf, nvl, 0, jn, i);
            wl[i] = acc;
            pn += acc * acc;
          }
        }
      }
      const double tt = sqrt(gm_block_sum2(pn, red, T));
      if (gm_opaque(threadIdx.x) < 64) {
        const int lane = gm_opaque(threadIdx.x);
        // previous rotations on the new column (KSPGMRESUpdateHessenberg): the
        // running entry obeys carry_(j+1) = -s_j carry_j + c_j h_(j+1), an
        // affine recurrence evaluated 64 rotations at a time by a DPP scan
        double carry = hcol[0];
        for (int base = 0; base < it; base += 64) {
          const int j = base + lane;
          const bool act = j < it;
          const double c = act ? lcc[j] : 1.0, sn = act ? lss[j] : 0.0, hn = act ? hcol[j + 1] : 0.0;
          double A = -sn, B = c * hn;
          gm_affine_scan(A, B);
          const double cnext = A * carry + B;            // carry_(j+1)
          const double cj = gm_shift_up1(cnext, carry);  // carry_j (lane 0: the carry in)
          if (act) hcol[j] = c * cj + sn * hn;
          carry = gm_readlane(cnext, min(63, it - 1 - base));
        }
        if (lane == 0) {
          hcol[it] = carry;
          hcol[it + 1] = tt;
          double hapbnd = fabs(tt / grs[it]);
          if (hapbnd > 1e-30) hapbnd = 1e-30;
          const int hap = tt < hapbnd;
          double res;
          if (!hap) {
            const double t1 = sqrt(hcol[it] * hcol[it] + hcol[it + 1] * hcol[it + 1]);
            const double c = hcol[it] / t1, sn = hcol[it + 1] / t1;
            lcc[it] = c;
            lss[it] = sn;
            grs[it + 1] = -sn * grs[it];
            grs[it] = c * grs[it];
            hcol[it] = c * hcol[it] + sn * hcol[it + 1];
            res = fabs(grs[it + 1]);
          } else {
            res = 0.0;
          }
          int rs = 0;
          if (res <= ttol) rs = 1;
          else if (res >= 1e4 * rn0) rs = -1;
          if (hap && !rs) rs = 1;
          s_flag[0] = rs;
          s_flag[1] = hap;
          s_val[0] = tt;
          s_val[1] = res;
        }
      }
      __syncthreads();
      reason = s_flag[0];
      const int hap = s_flag[1];
      for (int j = gm_opaque(threadIdx.x); j <= it + 1; j += T) a.H[(long)it * ld + j] = hcol[j];
      if (!hap) {
        const double inv = 1.0 / s_val[0];
        const bool keep = it + 1 < nvl;
        for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
          const double v1 = wl[i] * inv;
          vl[i] = v1;
          a.V[(long)(it + 1) * nf + i] = v1;
          if (keep) cache[(long)(it + 1) * nf + i] = v1;
        }
      }
      ++it;
      ++its;
      __syncthreads();
      if (reason || it >= kmax || its >= a.maxit) break;
    }
    // ---- KSPGMRESBuildSoln: back substitution on the rotated Hessenberg
    // (columns staged through the LDS cache, the serial sweep by one
    // wavefront), then x += V y
    const int top = it - 1;
    for (int j = gm_opaque(threadIdx.x); j <= top; j += T) yv[j] = grs[j];  // right-hand side, overwritten by y
    for (int k1 = top; k1 >= 0; k1 -= a.bsc) {
      const int k0 = k1 - a.bsc + 1 < 0 ? 0 : k1 - a.bsc + 1;
      const int nc = k1 - k0 + 1;
      __syncthreads();
      for (int q = gm_opaque(threadIdx.x); q < nc * (k1 + 1); q += T) {
        const int c = q / (k1 + 1), rr = q - c * (k1 + 1);
        cache[(long)c * ld + rr] = a.H[(long)(k0 + c) * ld + rr];
      }
      __syncthreads();
      if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        for (int k = k1; k >= k0; --k) {
          const double* col = cache + (long)(k - k0) * ld;
          const double yk = yv[k] / col[k];
          for (int j = lane; j < k; j += 64) yv[j] = yv[j] - col[j] * yk;
          if (lane == 0) yv[k] = yk;
          // LDS operations of one wavefront complete in order: the next
          // step's read of y(k-1) sees this step's update
          __builtin_amdgcn_wave_barrier();
        }
      }
    }
    __syncthreads();
    {
      const GmLayout g(gm_opaque(threadIdx.x), nf, T);
      if (nf <= T && g.nseg > 1) {
        const int per2 = (top + 1 + g.nseg - 1) / g.nseg;
        if (g.act) {
          const int q0 = min(top + 1, g.seg * per2), q1 = min(top + 1, q0 + per2);
          double acc = 0.0;  // sum_j y_j v_j[r] over this segment's j range
          for (int j = q0; j < q1; j += 8) {
            double v[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = a.V[(long)min(j + c, q1 - 1) * nf + g.r];
#pragma unroll
            for (int c = 0; c < 8; ++c)
              if (j + c < q1) acc += yv[j + c] * v[c];
          }
          part[g.seg * nf + g.r] = acc;
        }
        __syncthreads();
        for (int i = gm_opaque(threadIdx.x); i < nf; i += T) a.x[i] = a.x[i] + gm_sum_parts(part, nf, i, g.nseg);
      } else {
        for (int i = gm_opaque(threadIdx.x); i < nf; i += T) {
          double acc = 0.0;
          for (int j = 0; j <= top; ++j) acc += yv[j] * a.V[(long)j * nf + i];
          a.x[i] = a.x[i] + acc;
        }
      }
    }
    __syncthreads();
    if (reason) break;
    if (its >= a.maxit) {
      reason = -2;
      break;
    }
  }
  if (threadIdx.x == 0) {
    a.s->its = its;
    a.s->reason = reason;
    a.s->rn0 = rn0;
    a.s->ttol = ttol;
  }
}

// dynamic LDS of k_gmres_dense: vl, wl (nf each), hcol (kmax+2), lcc, lss
// (kmax each), grs, yv (kmax+1 each), part (kGmT), then the cache region
size_t gmres_dense_lds(int nf, int kmax, size_t cache_doubles) {
  return sizeof(double) * ((size_t)2 * nf + (size_t)5 * kmax + 4 + kGmT + cache_doubles);
}

bool gmres_dense_fits(int nf, int kmax, size_t max_lds) {
  return gmres_dense_lds(nf, kmax, (size_t)kmax + 1) + 1024 <= max_lds;
}

void gmres_dense(hipStream_t st, int nf, int kmax, int maxit, const double* S, const double* b, double* x, double* V,
                 double* H, GmresDev* s, double rtol, double atol, size_t max_lds) {
  // the cache takes what is left of the LDS: basis vectors during the
  // iterations, Hessenberg columns during the back substitution
  const size_t avail = max_lds > 1024 ? max_lds - 1024 : 0;  // room for the static shared arrays
  const size_t base = gmres_dense_lds(nf, kmax, 0);
  if (base + sizeof(double) * (kmax + 1) > avail) throw HipError("dense GMRES: restart too long for LDS");
  const size_t cache = (avail - base) / sizeof(double);
  const int nvl = (int)std::min<size_t>((size_t)kmax + 1, cache / (size_t)std::max(nf, 1));
  const int bsc = (int)std::max<size_t>(1, std::min<size_t>((size_t)kmax, cache / (size_t)(kmax + 1)));
  GmDenseArgs a{nf, kmax, maxit, nvl, bsc, S, b, x, V, H, s, rtol, atol};
  const size_t lds = gmres_dense_lds(nf, kmax, cache);
  hipLaunchKernelGGL(k_gmres_dense<24>, dim3(1), dim3(kGmT), lds, st, a);
  IB_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------
// The same dense solve spread over P workgroups of one XCD (k_gmres_coopw,
// below).  The launch has P workgroups per XCD, dealt by the dispatcher to
// the XCDs in turn; the P on the XCD the host names take part, so
// a solve keeps to one XCD's CUs and L2 and solves on different XCDs run side
// by side.  All waits are bounded: on a timeout the workgroups leave and the
// status stays at reason -3.
// ------------------------------------------------------------------------
constexpr long kCoopSpin = 1L << 22;

// The barrier block of a cooperative solve (unsigned words, cleared before
// each launch): word 0 the error flag, 8.. the workgroups' barrier counts,
// kXccSlot.. the XCD ids they publish, kClaimSlot the ranks claimed, kDoneSlot
// the workgroups that have ended their part.
constexpr int kCoopSyncDoubles = 40;
constexpr int kXccSlot = 40;
constexpr int kClaimSlot = 72;
constexpr int kDoneSlot = 73;
static_assert(kDoneSlot < 2 * kCoopSyncDoubles, "barrier block too small");

// The XCD this wavefront runs on (HW_REG_XCC_ID, bits 3:0).
__device__ __forceinline__ unsigned gw_xcc_id() { return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 0xFu; }

__global__ void k_xcc_probe(unsigned* ids) {
  if (threadIdx.x == 0) ids[blockIdx.x] = gw_xcc_id();
}

std::vector<int> gmres_xcc_ids(hipStream_t st) {
  static std::mutex mu;
  static std::map<int, std::vector<int>> known;
  int dev = 0;
  IB_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto it = known.find(dev);
  if (it != known.end()) return it->second;
  constexpr int kProbe = 64;
  unsigned* d = nullptr;
  IB_HIP(hipMalloc(&d, sizeof(unsigned) * kProbe));
  unsigned h[kProbe];
  hipLaunchKernelGGL(k_xcc_probe, dim3(kProbe), dim3(64), 0, st, d);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipFree(d);
  IB_HIP(e);
  std::vector<int> ids;
  for (unsigned v : h) ids.push_back((int)v);
  std::sort(ids.begin(), ids.end());
  ids.erase(std::unique(ids.begin(), ids.end()), ids.end());
  known[dev] = ids;
  return ids;
}

// v + the value of the lane 16 (32) further, modulo 32 (64): the rows of 16
// lanes (the halves of the wavefront) are swapped between two copies of v, and
// every lane adds the lower row's value and the higher's, so both lanes of a
// pair get the same bits
__device__ __forceinline__ double gm_add_xor16(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
  const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])) +
         __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
}
__device__ __forceinline__ double gm_add_xor32(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
  const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])) +
         __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
}

// Every lane of a wavefront holds partial sums v0..v3 of four rows; returns
// in lane l the sum over the 64 lanes of row ((l & 1) << 1) | ((l >> 1) & 1)
// (lanes 0, 1, 2, 3: rows 0, 2, 1, 3).  Pairs exchange half their rows
// (xor 1), then quads (xor 2), then the quads of a row of 16 are added
// (row_ror 4, 8) and the four rows of 16 (xor 16, 32).  Fixed order; the
// whole wavefront must be active.
__device__ __forceinline__ double gc_reduce4(double v0, double v1, double v2, double v3) {
  const int l = gm_opaque(threadIdx.x) & 63;
  const bool odd = l & 1, hi = l & 2;
  double k0 = odd ? v2 : v0, k1 = odd ? v3 : v1;
  const double s0 = odd ? v0 : v2, s1 = odd ? v1 : v3;
  k0 += gm_dpp<0xB1>(s0);
  k1 += gm_dpp<0xB1>(s1);
  double k = hi ? k1 : k0;
  k += gm_dpp<0x4E>(hi ? k0 : k1);
  k += gm_dpp<0x124>(k);
  k += gm_dpp<0x128>(k);
  return gm_add_xor32(gm_add_xor16(k));
}
// Wait until every vector memory operation this wavefront issued has
// completed; for the device-scope stores above that means they have
// reached the coherent level.  A workgroup-scope release fence does not
// emit this wait on gfx950 (it only orders within the CU), so without it
// another wavefront's flag store could overtake this wavefront's data.
__device__ __forceinline__ void gc_wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ------------------------------------------------------------------------
// The dense solve over P workgroups of one XCD: nf <= 1024 and Krylov spaces
// of up to 1023 vectors (full GMRES of the airfoil + flap system, nf = 800,
// restart 1000, over 32 workgroups; the hinged plate, nf = 202, over 4).
// Workgroup c owns rows [c R, c R + R) of S and of every Krylov vector:
//  * wavefront q owns RW local rows; lane l holds S[row][l + 64k], k < CQ, in
//    registers (nf <= 64 CQ), and the row sums go over the wavefront with DPP;
//  * the local rows of the basis are stored row-major in LDS (row r of
//    vector j at Vl[r NL + j]), so thread j forms the partial CGS coefficient
//    of vector j from conflict-free LDS reads, and the update w -= V h reads
//    consecutive j across the lanes; vectors j >= NL (past the LDS) are kept
//    in HBM in the same layout;
//  * only workgroup 0 keeps the Hessenberg matrix (in HBM, row by row) and
//    runs the back substitution at the end of a cycle.
// Systems of up to 256 entries take four rows per wavefront and few workgroups
// (the small form, RW = 4); it differs in the order of some sums and rotates
// each new column at once by an affine scan.
//
// What bounds it is latency: an Arnoldi step is a chain of small products
// joined by exchanges through L2.  So an exchanged value is its own flag: the
// buffers hold kUnset (a signalling NaN, which no arithmetic result is) where
// nothing has been published, a reader polls the value itself until it is
// there, and no barrier, store wait or second load stands between a
// workgroup's last product and its neighbours' next one.  A step has three
// exchanges: the partial CGS coefficients (x1), their sums (x2: workgroup c
// sums coefficients c, c + P, ...; left out while every workgroup can load
// all partials in two loads per thread) and the rows of the new vector u
// (x3).  Everything that is not on that chain runs beside it:
//  * every workgroup has the whole of the new vector u, exchanged
//    unnormalised, so |u| is its own last wavefront's, the same bits
//    everywhere, while the others form S u (S v = S u / |u|; the small form
//    multiplies v itself, after |u|);
//  * the Givens step and the stopping tests are the last wavefront's too,
//    while the others form the dot products of S v.  A step's coefficients are
//    therefore on their way before it is known whether the step before
//    converged; after the last one they are not used;
//  * entry it of the new column after the previous rotations is
//    sum_j alpha_j h_j with alpha updated as [-s_it alpha, c_it], one dot
//    product; the stored columns are rotated at the cycle's end (small form:
//    the scan, beside the update).
// Each buffer has three copies, used in turn.  A workgroup clears what it
// published in step s once it has published its rows of step s + 1 (its x2 of
// that step was complete, which takes every workgroup's x1 of step s + 1, and
// each published that after it had read all of step s), and waits for these
// stores before it publishes its rows of step s + 2; a reader comes back to
// the copy in step s + 3, after it has read all rows of step s + 2.  The clears
// thus run while the rows of step s + 1 travel.
//
// Microseconds per Arnoldi step (events around the launches, start-up and
// back substitution included), with grid barriers around each exchange and
// now: airfoil + flap (nf = 800, ~460 steps a solve) 9.38 -> 6.55; plate (nf =
// 202) 6.74 -> 5.23; flexible plate 6.69 -> 5.26; GMRES(30) of the cylinder
// (nf = 314) 5.99 -> 3.55; a 42-entry system 5.77 -> 4.28.  Both layouts round
// as the kernels with grid barriers did (the solution's bits are theirs).
// ------------------------------------------------------------------------
constexpr int kCwBlk = 32;
constexpr int kCwLd = kCwBlk + 1;  // row stride of a staged block (no bank conflicts down a column)
constexpr unsigned long long kUnset = 0x7ff4c0de5eed0001ull;

struct GmCoopWArgs {
  int nf, kmax, maxit, P, lPg, R, NL;  // Pg = 2^lPg: the power of two >= P
  int xcd;  // the XCD whose workgroups take part (-1: workgroups 0, 8, 16, ...)
  int l2x;  // 1: exchange through one XCD's L2 when every workgroup is found there
  int fail_rank;  // the workgroup that takes its last wait of a cycle as timed out (-1: none)
  const double* S;
  const double* b;
  double* x;
  GmresDev* s;
  double rtol, atol;
  unsigned* sync;  // [0] error, [8 + c] barriers passed by workgroup c
  double* x1;      // 3 x (kmax + 1) x Pg: partial CGS coefficients, coefficient j of workgroup q at j Pg + q
  double* x2;      // 3 x (kmax + 1): summed CGS coefficients
  double* x3;      // 3 x nf: the new vector, unnormalised
  double* rfull;   // nf: the residual at a cycle's start
  double* norms;   // P x 2: partial squared norms of r and b
  double* yg;      // kmax + 1: the back substitution's y
  double* Ht;      // (kmax + 1) x kmax: the Hessenberg matrix, entry (j, k) at j kmax + k
  double* rot;     // 3 kmax: the rotations and the rotated diagonal, (c_k, s_k, d_k) at 3k
  double* Vg;      // P x R x (kmax + 1 - NL): basis vectors NL.. of each workgroup's rows
};

// Every lane holds partial sums v0, v1 of two rows; returns in lane 0 the
// sum over the 64 lanes of row 0 and in lane 1 that of row 1.  Pairs swap
// a row (xor 1), then the pairs of a quad are added (xor 2), the quads of a
// row of 16 (row_ror 4, 8) and the four rows of 16 (xor 16, 32).  Fixed
// order; the whole wavefront must be active.
__device__ __forceinline__ double gw_reduce2(double v0, double v1) {
  const int l = gm_opaque(threadIdx.x) & 63;
  const bool odd = l & 1;
  double k = odd ? v1 : v0;
  k += gm_dpp<0xB1>(odd ? v0 : v1);
  k += gm_dpp<0x4E>(k);
  k += gm_dpp<0x124>(k);
  k += gm_dpp<0x128>(k);
  return gm_add_xor32(gm_add_xor16(k));
}
// the same for RW = 2 or 4 rows; lane l < RW gets the sum of row gw_row<RW>(l)
template <int RW>
__device__ __forceinline__ double gw_reduce_rows(const double (&v)[RW]) {
  if constexpr (RW == 2) return gw_reduce2(v[0], v[1]);
  else return gc_reduce4(v[0], v[1], v[2], v[3]);
}
template <int RW>
__device__ __forceinline__ int gw_row(int l) {
  if constexpr (RW == 2) return l & 1;
  else return ((l & 1) << 1) | ((l >> 1) & 1);
}

// Butterfly sum over aligned groups of g = 1, 2, 4, ..., 32 consecutive
// lanes: xor 1 and xor 2 through DPP quad permutes; then, since all lanes of a
// quad (of 8 lanes) hold the same bits, xor 4 (8) as a mirror of 8 (16)
// lanes, and xor 16 by swapping rows.  Every lane of a group ends with the
// same bits, ((p0 + p1) + (p2 + p3)) + ... in one fixed order.  The whole
// wavefront must be active.
__device__ __forceinline__ double gw_group_sum(double p, int g) {
  if (g >= 2) p += gm_dpp<0xB1>(p);
  if (g >= 4) p += gm_dpp<0x4E>(p);
  if (g >= 8) p += gm_dpp<0x141>(p);
  if (g >= 16) p += gm_dpp<0x140>(p);
  if (g >= 32) p = gm_add_xor16(p);
  return p;
}

// Lanes per CGS coefficient in the dot phase of step it (its logarithm): as
// many as the 1024 threads allow, up to 8 (groups never straddle a wavefront).
__device__ __forceinline__ int gw_log_lanes_per_coef(int it) {
  const int n = it + 1;
  return 8 * n <= kGmT ? 3 : (4 * n <= kGmT ? 2 : (2 * n <= kGmT ? 1 : 0));
}

// gm_block_sum2 without its 16 loads in flight (they would cost the solve the
// registers that hold S)
__device__ __forceinline__ double gw_block_sum(double v, double* red) {
  const int t = gm_opaque(threadIdx.x);
  v = gm_wave_sum(v);
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  double tot = 0.0;
#pragma unroll 1
  for (int q = 0; q < kGmT / 64; ++q) tot += red[q];
  __syncthreads();
  return tot;
}

// the sum over lanes 0..n-1 in that order (the whole wavefront must be active)
__device__ __forceinline__ double gw_seq_sum(double v, int n) {
  double t = 0.0;
  for (int q = 0; q < n; ++q) t += gm_readlane(v, q);
  return t;
}

// a product rounded by itself, whatever it is added to
__device__ __forceinline__ double gw_mul(double a, double b) {
#pragma clang fp contract(off)
  return a * b;
}

// Exchange between the workgroups of a cooperative solve.  Loads are
// device-scope atomic loads: they bypass the CU's L1 and are served by L2
// (measured on MI355X: ~90 ns per dependent load, against ~56 ns for an L1
// hit); an atomic load is always a vector memory access, where a plain load
// of a uniform address could be served by the scalar cache.  Stores: device
// scope, coherent across XCDs, or with X2 (every workgroup on one XCD, checked
// at the start of the launch) workgroup-scope stores, which complete at that
// XCD's L2 -- the one L2 every load of the exchange reads -- instead of at
// memory.
__device__ __forceinline__ double xc_ld(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool X2>
__device__ __forceinline__ void xc_st_bits(double* p, unsigned long long v) {
  unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
  if constexpr (X2) __hip_atomic_store(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else __hip_atomic_store(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool X2>
__device__ __forceinline__ void xc_st(double* p, double v) {
  xc_st_bits<X2>(p, (unsigned long long)__double_as_longlong(v));
}
// publishes a value that others poll; any NaN becomes the quiet one, so that
// it is never taken for kUnset
template <bool X2>
__device__ __forceinline__ void xc_put(double* p, double v) {
  xc_st_bits<X2>(p, v == v ? (unsigned long long)__double_as_longlong(v) : 0x7ff8000000000000ull);
}
__device__ __forceinline__ unsigned xc_ldu(const unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool X2>
__device__ __forceinline__ void xc_stu(unsigned* p, unsigned v) {
  if constexpr (X2) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether a wavefront that has polled n times gives up: after kCoopSpin polls,
// or when another wavefront or workgroup has.  The error words are then set,
// the wavefront goes on with what it has, and the workgroup leaves at its next
// check of s_err.
__device__ __forceinline__ bool xc_give_up(long n, unsigned* err, int* s_err) {
  if ((n & 63) != 0 || (n <= kCoopSpin && xc_ldu(err) == 0u && *(volatile int*)s_err == 0)) return false;
  if ((threadIdx.x & 63) == 0) {
    __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *(volatile int*)s_err = 1;
  }
  return true;
}

// The published value at p for the lanes that need one (0 for the others):
// the wavefront polls until all of them are there.  The whole wavefront must
// be active.
__device__ __forceinline__ double xc_poll(const double* p, bool need, unsigned* err, int* s_err) {
  unsigned long long v = 0;
  long n = 0;
  while (true) {
    if (need)
      v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__all(!need || v != kUnset)) break;
    if (xc_give_up(++n, err, s_err)) break;
  }
  return __longlong_as_double((long long)v);
}

// Two published values, polled together.
__device__ __forceinline__ double2 xc_poll2(const double* p0, bool need0, const double* p1, bool need1, unsigned* err,
                                            int* s_err) {
  unsigned long long v0 = 0, v1 = 0;
  long n = 0;
  while (true) {
    if (need0)
      v0 = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (need1)
      v1 = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__all((!need0 || v0 != kUnset) && (!need1 || v1 != kUnset))) break;
    if (xc_give_up(++n, err, s_err)) break;
  }
  return make_double2(__longlong_as_double((long long)v0), __longlong_as_double((long long)v1));
}

// Grid barrier number k (1, 2, ...) over the P workgroups, for the few
// exchanges outside the Arnoldi steps.  Every wavefront waits for its own
// stores to complete (gc_wait_stores) before the workgroup barrier, so when
// wavefront 0 then publishes flag[c] = k every store of workgroup c is
// visible to the others' loads; wavefront 0 polls the P flags (one lane each)
// until all have reached k, and the others wait at the second workgroup
// barrier.  Bounded: on a timeout (or another workgroup's) the error word is
// set and every workgroup leaves.
template <bool X2>
__device__ __forceinline__ bool xc_sync(unsigned* sync, int P, int c, unsigned k, int* s_err) {
  gc_wait_stores();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __syncthreads();
  if (threadIdx.x < 64) {
    unsigned* err = sync;
    unsigned* fl = sync + 8;
    const int lane = threadIdx.x;
    if (lane == 0) xc_stu<X2>(fl + c, k);
    long n = 0;
    while (true) {
      const unsigned v = lane < P ? xc_ldu(fl + lane) : k;
      if (__all(v >= k)) break;
      if (xc_ldu(err) != 0u || ++n > kCoopSpin) {
        if (lane == 0) {
          __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          *s_err = 1;
        }
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  __syncthreads();
  return *s_err == 0;
}

// Sets what workgroup c published in a step of n coefficients to kUnset, in
// copy k of the buffers (threads t, t + nthr, ...).
template <bool X2>
__device__ __forceinline__ void coopw_clear(const GmCoopWArgs& a, int c, int r0, int Rc, int k, int n, int t, int nthr) {
  double* x1 = a.x1 + ((k * (a.kmax + 1)) << a.lPg) + c;
  double* x2 = a.x2 + k * (a.kmax + 1);
  for (int j = t; j < n; j += nthr) xc_st_bits<X2>(x1 + (j << a.lPg), kUnset);
  for (int j = c + t * a.P; j < n; j += nthr * a.P) xc_st_bits<X2>(x2 + j, kUnset);
  for (int r = t; r < Rc; r += nthr) xc_st_bits<X2>(a.x3 + k * a.nf + r0 + r, kUnset);
}

template <int RW, int CQ, bool X2>
__device__ __forceinline__ void coopw_solve(const GmCoopWArgs& a, int c, unsigned bk, double* dyn, double* red,
                                            double* s_val, int* s_flag, int* s_err) {
  constexpr bool kSmall = RW == 4;
  const int nf = a.nf, kmax = a.kmax, ld = kmax + 1, T = kGmT, R = a.R, NL = a.NL, P = a.P, lPg = a.lPg, Pg = 1 << lPg;
  const int r0 = c * R, Rc = min(nf, r0 + R) - r0;
  const int ldg = ld - NL;  // row stride of the basis vectors kept in HBM
  double* Vgc = a.Vg + (size_t)c * R * (size_t)max(ldg, 0);
  double* wl = dyn;                    // 64: local rows of S u
  double* nrm = wl + 64;               // 32: the workgroups' shares of |u|^2
  double* hcol = nrm + 32;             // kmax + 2: CGS coefficients of S u (y at a cycle's end)
  double* alpha = hcol + kmax + 2;     // kmax + 2: entry it of the rotated column = sum_j alpha_j h_j
  double* grs = alpha + kmax + 2;      // kmax + 1 (y of the back substitution in place)
  double* stg = grs + kmax + 1;        // kCwBlk x kCwLd: a diagonal block of the back substitution
  double* ub = stg + kCwBlk * kCwLd;   // nf: the vector of a product, u
  double* lss = ub + nf;               // small form, kmax: the rotations' sines (their cosines in alpha)
  double* Vl = lss + (kSmall ? kmax : 0);  // R NL: local rows of basis vectors 0..NL-1, row-major
  // rows RW wq .. of S, columns ln + 64 k, in registers (0 outside the matrix)
  double s[RW][CQ];
  {
    const int wq = threadIdx.x >> 6, ln = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < RW; ++i)
#pragma unroll
      for (int k = 0; k < CQ; ++k) {
        const int row = RW * wq + i, col = ln + 64 * k;
        s[i][k] = row < Rc && col < nf ? a.S[(long)col * nf + r0 + row] : 0.0;
      }
  }
  __syncthreads();

  // wl = S[local rows] ub (small form: ub times scale) (wavefront q: rows RW q ..)
  auto matvec = [&](double scale) {
    const int q = gm_opaque(threadIdx.x) >> 6, l = gm_opaque(threadIdx.x) & 63;
    if (RW * q < Rc) {  // uniform over the wavefront
      double v[CQ], acc[RW];
#pragma unroll
      for (int k = 0; k < CQ; ++k) v[k] = kSmall ? gw_mul(ub[min(l + 64 * k, nf - 1)], scale) : ub[min(l + 64 * k, nf - 1)];
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        acc[i] = 0.0;
#pragma unroll
        for (int k = 0; k < CQ; ++k) acc[i] += s[i][k] * v[k];  // s is 0 past the matrix
      }
      const double sum = gw_reduce_rows<RW>(acc);
      const int row = RW * q + gw_row<RW>(l);
      if (l < RW && row < Rc) wl[row] = sum;
    }
  };
  // acc[i] += sum_{j = l, l + 64, ... < jn} coef[j] V(RW q + i, j): four
  // chunks of 64 vectors in flight while all are in LDS (terms past jn add 0)
  auto rows_dot = [&](const double* coef, int jn, int q, int l, double (&acc)[RW]) {
    int rr[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) rr[i] = min(RW * q + i, Rc - 1) * NL;
    if (jn <= NL) {
#pragma unroll 1
      for (int w = 0; w < jn; w += 256) {
        double h[4], v[4][RW];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int j = min(w + 64 * b + l, jn - 1);
          h[b] = coef[j];
#pragma unroll
          for (int i = 0; i < RW; ++i) v[b][i] = Vl[rr[i] + j];
        }
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int i = 0; i < RW; ++i) acc[i] += (w + 64 * b + l < jn ? h[b] : 0.0) * v[b][i];
      }
      return;
    }
#pragma unroll 1
    for (int j = l; j < jn; j += 64) {
      const double h = coef[j];
#pragma unroll
      for (int i = 0; i < RW; ++i)
        acc[i] += h * (j < NL ? Vl[rr[i] + j] : Vgc[(size_t)min(RW * q + i, Rc - 1) * ldg + (j - NL)]);
    }
  };

  int its = 0, reason = 0, first = 1;
  double rn0 = 0.0, ttol = 0.0;
  bool ok = true;
  while (true) {
    // ---- cycle start: r = b - S x (x from every workgroup's rows)
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) ub[i] = xc_ld(a.x + i);
    __syncthreads();
    matvec(1.0);
    __syncthreads();
    double pr = 0.0, pb = 0.0;
    for (int r = gm_opaque(threadIdx.x); r < Rc; r += T) {
      const double bv = a.b[r0 + r];
      const double rv = bv - wl[r];
      xc_st<X2>(a.rfull + r0 + r, rv);
      pr += rv * rv;
      pb += bv * bv;
    }
    pr = gw_block_sum(pr, red);
    pb = gw_block_sum(pb, red);
    if (threadIdx.x == 0) {
      xc_st<X2>(a.norms + c * 2, pr);
      xc_st<X2>(a.norms + c * 2 + 1, pb);
    }
    if (!xc_sync<X2>(a.sync, P, c, ++bk, s_err)) break;
    if (threadIdx.x < 64) {
      const int lane = threadIdx.x;
      const double nr = lane < P ? xc_ld(a.norms + lane * 2) : 0.0, nb = lane < P ? xc_ld(a.norms + lane * 2 + 1) : 0.0;
      const double sr = kSmall ? gw_seq_sum(nr, P) : gm_wave_sum(nr), sb = kSmall ? gw_seq_sum(nb, P) : gm_wave_sum(nb);
      if (lane == 0) {
        s_val[0] = sr;
        s_val[1] = sb;
      }
    }
    for (int i = gm_opaque(threadIdx.x); i < nf; i += T) ub[i] = xc_ld(a.rfull + i);
    __syncthreads();
    const double res0 = sqrt(s_val[0]), bn = sqrt(s_val[1]);
    if (first) {
      rn0 = bn > 0.0 ? bn : res0;
      ttol = fmax(a.rtol * rn0, a.atol);
      first = 0;
    }
    if (res0 == 0.0 || res0 <= ttol) reason = 1;
    else if (res0 >= 1e4 * rn0) reason = -1;
    if (reason) break;
    if constexpr (kSmall)
      for (int i = gm_opaque(threadIdx.x); i < nf; i += T) ub[i] = ub[i] / res0;
    __syncthreads();  // s_val is rewritten below
    int it = 0;         // columns formed
    int cur = 0, old = 2;  // it mod 3, (it - 1) mod 3
    double hv = 0.0;    // last wavefront: entry it - 1 of column it - 1 after the previous rotations
    double cc = 1.0, sn = 0.0;  // last wavefront: the rotation of column it - 1
    while (true) {
      // here ub = u, the unnormalised vector v_it
      const bool more = it < kmax && its < a.maxit;
      double tt = res0;  // last wavefront: |u|
      if constexpr (!kSmall) matvec(1.0);
      if (gm_opaque(threadIdx.x) >= T - 64) {
        const int lane = gm_opaque(threadIdx.x) & 63;
        if (it > 0) {
          if constexpr (kSmall) {
            // per workgroup its wavefronts' shares (stg) in turn, then the workgroups'
            double v[16], t = 0.0;
#pragma unroll
            for (int q = 0; q < 16; ++q) v[q] = stg[16 * min(lane, P - 1) + q];
#pragma unroll
            for (int q = 0; q < 16; ++q) t += v[q];
            tt = sqrt(gw_seq_sum(t, P));
          } else {
            tt = sqrt(gm_wave_sum(lane < P ? nrm[lane] : 0.0));
          }
        }
        // the small form divides the residual itself (its u at it = 0 is v_0)
        if (lane == 0) s_val[0] = kSmall && it == 0 ? 1.0 : 1.0 / tt;
      }
      if constexpr (kSmall) {
        __syncthreads();
        matvec(s_val[0]);
      }
      if (threadIdx.x == 0) s_flag[2] = *(volatile int*)s_err;
      __syncthreads();
      if (s_flag[2]) {
        ok = false;
        break;
      }
      const double inv = s_val[0];  // v_it = u inv, S v_it = (S u) inv
      // partial CGS coefficients <S v_it, v_j>, j <= it, over the local
      // rows: g lanes per j, lane sub takes rows sub, sub + g, ...; blocks of
      // four rows, the loads of a block ahead of its sums (the rows past Rc
      // add 0)
      if constexpr (kSmall) {
        // 16 lanes per coefficient, up to four rows each
        if (more) {
          const int t = gm_opaque(threadIdx.x), sub = t & 15;
          double w[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) w[q] = wl[min(sub + 16 * q, Rc - 1)];
          for (int j0 = 0; j0 + ((t & ~63) >> 4) <= it; j0 += T / 16) {  // uniform over the wavefront
            const int j = j0 + (t >> 4);
            const double* vl = j < it ? Vl + j : ub + r0;  // v_it is not stored yet
            const int ldv = j < it ? NL : 1;
            const double sc = j < it ? 1.0 : inv;
            double p = 0.0;
            if (j <= it) {
              double v[4];
#pragma unroll
              for (int q = 0; q < 4; ++q) v[q] = vl[min(sub + 16 * q, Rc - 1) * ldv];
#pragma unroll
              for (int q = 0; q < 4; ++q) p += (sub + 16 * q < Rc ? w[q] : 0.0) * gw_mul(v[q], sc);
            }
            p = gm_row_sum16(p);
            if (j <= it && sub == 0) xc_put<X2>(a.x1 + ((cur * ld + j) << lPg) + c, p);
          }
        }
      } else if (more) {
        const int lg = gw_log_lanes_per_coef(it), g = 1 << lg;
        const int t = gm_opaque(threadIdx.x), j = t >> lg, sub = t & (g - 1);
        if (((t & ~63) >> lg) <= it) {  // uniform over the wavefront
          double p = 0.0;
          if (j < it && j >= NL) {
            const double* vg = Vgc + (j - NL);
#pragma unroll 1
            for (int r1 = sub; r1 < Rc; r1 += 4 * g) {
              double w[4], v[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int rr = min(r1 + (i << lg), Rc - 1);
                w[i] = wl[rr];
                v[i] = vg[(size_t)rr * ldg];
              }
#pragma unroll
              for (int i = 0; i < 4; ++i) p += (r1 + (i << lg) < Rc ? gw_mul(w[i], inv) : 0.0) * v[i];
            }
          } else if (j <= it) {
            const double* vl = j < it ? Vl + j : ub + r0;  // v_it is not stored yet
            const int ldv = j < it ? NL : 1;
            const double sc = j < it ? 1.0 : inv;
#pragma unroll 1
            for (int r1 = sub; r1 < Rc; r1 += 4 * g) {
              double w[4], v[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int rr = min(r1 + (i << lg), Rc - 1);
                w[i] = wl[rr];
                v[i] = vl[rr * ldv];
              }
#pragma unroll
              for (int i = 0; i < 4; ++i)
                p += (r1 + (i << lg) < Rc ? gw_mul(w[i], inv) : 0.0) * gw_mul(v[i], sc);
            }
          }
          p = gw_group_sum(p, g);
          if (j <= it && sub == 0) xc_put<X2>(a.x1 + ((cur * ld + j) << lPg) + c, p);
        }
      }
      if (gm_opaque(threadIdx.x) >= T - 64) {
        // the last wavefront: the Givens step of column k = it - 1
        // (KSPGMRESUpdateHessenberg)
        const int lane = gm_opaque(threadIdx.x) & 63;
        int rs = 0;
        cc = 1.0;
        sn = 0.0;
        if (it == 0) {
          if (lane == 0) grs[0] = res0;
        } else {
          const int k = it - 1;
          const double gk = grs[k];
          // tt < min(|tt / grs[k]|, 1e-30) is a happy breakdown (the
          // quotient is needed only when tt < 1e-30)
          const bool hap = tt < 1e-30 && tt < fabs(tt / gk);
          double res = 0.0, diag = hv;
          if (!hap) {
            const double t1 = sqrt(kSmall ? __builtin_fma(tt, tt, gw_mul(hv, hv)) : __builtin_fma(hv, hv, gw_mul(tt, tt)));
            cc = hv / t1;
            sn = tt / t1;
            diag = cc * hv + sn * tt;
            res = fabs(sn * gk);
          }
          if (res <= ttol) rs = 1;
          else if (res >= 1e4 * rn0) rs = -1;
          if (hap && !rs) rs = 1;
          if (lane == 0) {
            if (!hap) {
              grs[it] = -sn * gk;
              grs[k] = cc * gk;
            }
            if constexpr (kSmall) {
              alpha[k] = cc;
              lss[k] = sn;
              if (c == 0) a.Ht[(long)k * kmax + k] = diag;
            } else if (c == 0) {
              a.rot[3 * k] = cc;
              a.rot[3 * k + 1] = sn;
              a.rot[3 * k + 2] = diag;
            }
          }
        }
        if (lane == 0) s_flag[0] = rs;
      }
      if (more) {
        const int n = it + 1;
        const double* x1 = a.x1 + ((cur * ld) << lPg);  // below 2^17
        if constexpr (kSmall) {
          // every workgroup sums the partials of all (thread j coefficient j)
          const int j = gm_opaque(threadIdx.x);
          if ((j & ~63) < n) {  // uniform over the wavefront
            const double* xj = x1 + (j << lPg);
            double h = 0.0;
            for (int q = 0; q < P; q += 2) {
              const double2 v = xc_poll2(xj + q, j < n, xj + q + 1, j < n && q + 1 < P, a.sync, s_err);
              h += v.x;
              if (q + 1 < P) h += v.y;
            }
            if (j < n) hcol[j] = h;
          }
        } else if ((n << lPg) <= 2 * T) {
          // few partials: every workgroup sums all of them (Pg lanes per
          // coefficient, fixed butterfly)
          for (int base = 0; base < (n << lPg); base += T) {
            const int i = base + gm_opaque(threadIdx.x), j = i >> lPg, q = i & (Pg - 1);
            if (((i & ~63) >> lPg) >= n) break;  // uniform over the wavefront
            const double h = gw_group_sum(xc_poll(x1 + i, j < n && q < P, a.sync, s_err), Pg);
            if (j < n && q == 0) hcol[j] = h;
          }
        } else {
          // workgroup c sums coefficients c, c + P, ... in the same way and
          // publishes the sums; each partial is read once
          for (int base = 0; c + base * P < n; base += T >> lPg) {
            const int t = gm_opaque(threadIdx.x), jj = base + (t >> lPg), q = t & (Pg - 1);
            const int j = c + jj * P;
            if (c + (base + ((t & ~63) >> lPg)) * P >= n) break;  // uniform over the wavefront
            const double h = gw_group_sum(xc_poll(x1 + (j << lPg) + q, j < n && q < P, a.sync, s_err), Pg);
            if (j < n && q == 0) xc_put<X2>(a.x2 + cur * ld + j, h);
          }
          const int t = gm_opaque(threadIdx.x);  // n <= kmax + 1 <= T
          if ((t & ~63) < n) {  // uniform over the wavefront
            const double h = xc_poll(a.x2 + cur * ld + t, t < n, a.sync, s_err);
            if (t < n) hcol[t] = h;
          }
        }
      }
      __syncthreads();
      reason = s_flag[0];
      if (reason || !more) break;
      // the new vector's local rows, S v_it - sum_j h_j v_j
      {
        const int q = gm_opaque(threadIdx.x) >> 6, l = gm_opaque(threadIdx.x) & 63;
        if (RW * q < Rc) {  // uniform over the wavefront
          double acc[RW];
#pragma unroll
          for (int i = 0; i < RW; ++i) acc[i] = 0.0;
          rows_dot(hcol, it, q, l, acc);
          if (l == (it & 63)) {  // the term of v_it, the last of its lane
            const double h = hcol[it];
#pragma unroll
            for (int i = 0; i < RW; ++i) acc[i] += h * gw_mul(ub[r0 + min(RW * q + i, Rc - 1)], inv);
          }
#pragma unroll
          for (int i = 0; i < RW; ++i) acc[i] = -acc[i];
          // this lane's row, read before the wait and the store below: once a
          // workgroup's rows are out, its polling wavefronts may write the next
          // vector over ub
          const int row = RW * q + gw_row<RW>(l), rr = min(row, Rc - 1);
          const double v = gw_mul(ub[r0 + rr], inv), w = kSmall ? wl[rr] : gw_mul(wl[rr], inv);
          const double sum = gw_reduce_rows<RW>(acc);
          gc_wait_stores();  // the clears of the step before
          if (l < RW && row < Rc) {
            xc_put<X2>(a.x3 + cur * nf + r0 + row, w + sum);
            if (it < NL) Vl[row * NL + it] = v;
            else Vgc[(size_t)row * ldg + (it - NL)] = v;
          }
          // what step it - 1 published
          if (it > 0)
            coopw_clear<X2>(a, c, r0, Rc, old, it, gm_opaque(threadIdx.x), 64 * ((Rc + RW - 1) / RW));
        }
      }
      if (gm_opaque(threadIdx.x) >= T - 64) {
        const int lane = gm_opaque(threadIdx.x) & 63;
        if constexpr (kSmall) {
          // the previous rotations applied to the new column as an
          // affine-recurrence scan, 64 rotations at a time
          double carry = hcol[0];
          for (int base = 0; base < it; base += 64) {
            const int j = base + lane;
            const bool act = j < it;
            const double cj0 = act ? alpha[j] : 1.0, sj = act ? lss[j] : 0.0, hn = act ? hcol[j + 1] : 0.0;
            double A = -sj, B = cj0 * hn;
            gm_affine_scan(A, B);
            const double cnext = A * carry + B;
            const double cj = gm_shift_up1(cnext, carry);
            if (act && c == 0) a.Ht[(long)j * kmax + it] = cj0 * cj + sj * hn;
            carry = gm_readlane(cnext, min(63, it - 1 - base));
          }
          hv = carry;
        } else {
          double part = 0.0;  // lane w: the sum over j = 64 w ..
#pragma unroll 1
          for (int w0 = 0; 64 * w0 <= it; w0 += 4) {
            double p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = 64 * (w0 + i) + lane, jj = min(j, it);
              double al = alpha[jj];
              const double h = hcol[jj];
              al = j < it ? -sn * al : cc;
              if (j <= it) alpha[j] = al;
              p[i] = j <= it ? gw_mul(al, h) : 0.0;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const double q = gm_wave_sum(p[i]);
              if (lane == w0 + i) part = q;
            }
          }
          hv = gm_readlane(gm_row_sum16(part), 0);
        }
      }
      if (!kSmall && c == 0) {
        for (int j = gm_opaque(threadIdx.x); j <= it; j += T) a.Ht[(long)j * kmax + it] = hcol[j];
      }
      ++it;
      ++its;
      old = cur;
      cur = cur == 2 ? 0 : cur + 1;
      // the new vector, RW adjacent rows of a workgroup per lane (16 lanes a
      // workgroup), and the workgroups' shares of its squared norm: the
      // squares of the rows a wavefront owns, then gm_row_sum16 over the
      // wavefronts (small form: one after the other, below)
      {
        const int t = gm_opaque(threadIdx.x), cq = t >> 4;
        if ((t >> 6) * 4 < P) {  // uniform over the wavefront
          const int rend = cq < P ? min(cq * R + R, nf) : 0;
          const int ra = cq * R + RW * (t & 15);
          const double* p = a.x3 + old * nf + ra;
          const double2 u = xc_poll2(p, ra < rend, p + 1, ra + 1 < rend, a.sync, s_err);
          if (ra < rend) ub[ra] = u.x;
          if (ra + 1 < rend) ub[ra + 1] = u.y;
          if constexpr (kSmall) {
            const double2 v = xc_poll2(p + 2, ra + 2 < rend, p + 3, ra + 3 < rend, a.sync, s_err);
            if (ra + 2 < rend) ub[ra + 2] = v.x;
            if (ra + 3 < rend) ub[ra + 3] = v.y;
            if (cq < P)
              stg[t] = (gw_mul(u.x, u.x) + gw_mul(v.x, v.x)) + (gw_mul(u.y, u.y) + gw_mul(v.y, v.y));
          } else {
            const double tot = gm_row_sum16(gw_mul(u.x, u.x) + gw_mul(u.y, u.y));
            if ((t & 15) == 0 && cq < P) nrm[cq] = tot;
          }
        }
      }
      __syncthreads();
    }
    if (!ok) break;
    if (c == a.fail_rank && threadIdx.x == 0) {  // as xc_give_up in the last step
      __hip_atomic_store(a.sync, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *s_err = 1;
    }
    // ---- KSPGMRESBuildSoln: workgroup 0 rotates the columns, solves the
    // triangular system (grs becomes y in place) and publishes y
    const int top = it - 1;
    if (c == 0) {
      if constexpr (!kSmall) {
        double* rc = hcol;   // the rotations (hcol and alpha are free here)
        double* rsn = alpha;
        for (int k = gm_opaque(threadIdx.x); k <= top; k += T) {
          rc[k] = a.rot[3 * k];
          rsn[k] = a.rot[3 * k + 1];
        }
        __syncthreads();
        // the previous rotations on every column k (thread k), its diagonal
        // from the step: the rows are read across the columns, eight rows
        // ahead of the recurrence
        for (int k = gm_opaque(threadIdx.x); k <= top; k += T) {
          double* col = a.Ht + k;
          double carry = col[0];
          for (int j0 = 0; j0 < k; j0 += 8) {
            double h[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) h[i] = col[(long)min(j0 + i + 1, k) * kmax];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int j = j0 + i;
              if (j < k) {
                const double hn = h[i];
                col[(long)j * kmax] = rc[j] * carry + rsn[j] * hn;
                carry = -rsn[j] * carry + rc[j] * hn;
              }
            }
          }
          col[(long)k * kmax] = a.rot[3 * k + 2];
        }
      }
      __syncthreads();
      for (int kb1 = top; kb1 >= 0; kb1 -= kCwBlk) {
        const int kb0 = max(0, kb1 - kCwBlk + 1), nb = kb1 - kb0 + 1;
        // row i, column k of the diagonal block at i kCwLd + k
        {
          const int i = gm_opaque(threadIdx.x) / kCwBlk, k = gm_opaque(threadIdx.x) % kCwBlk;
          if (k < nb && i <= k) stg[i * kCwLd + k] = a.Ht[(long)(kb0 + i) * kmax + kb0 + k];
        }
        __syncthreads();
        if (threadIdx.x < 64) {
          const int lane = threadIdx.x;
          double ti = lane < nb ? grs[kb0 + lane] : 0.0;
          for (int k = nb - 1; k >= 0; --k) {
            const double yk = gm_readlane(ti, k) / stg[k * kCwLd + k];
            if (lane < k) ti -= stg[lane * kCwLd + k] * yk;
            if (lane == k) ti = yk;
          }
          if (lane < nb) grs[kb0 + lane] = ti;
        }
        __syncthreads();
        // the rows above the block, columns of the block in descending
        // order, eight loads ahead
        for (int i = gm_opaque(threadIdx.x); i < kb0; i += T) {
          const double* row = a.Ht + (long)i * kmax + kb0;
          double t = grs[i];
          for (int k0 = nb - 1; k0 >= 0; k0 -= 8) {
            double h[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) h[q] = row[max(k0 - q, 0)];
#pragma unroll
            for (int q = 0; q < 8; ++q)
              if (k0 - q >= 0) t -= h[q] * grs[kb0 + k0 - q];
          }
          grs[i] = t;
        }
        __syncthreads();
      }
      for (int j = gm_opaque(threadIdx.x); j <= top; j += T) xc_st<X2>(a.yg + j, grs[j]);
    }
    if (!xc_sync<X2>(a.sync, P, c, ++bk, s_err)) break;
    for (int j = gm_opaque(threadIdx.x); j <= top; j += T) hcol[j] = xc_ld(a.yg + j);
    __syncthreads();
    // x += V y on the local rows
    if constexpr (kSmall) {
      const int r = gm_opaque(threadIdx.x);
      if (r < Rc) {
        double acc = 0.0;
        for (int j0 = 0; j0 <= top; j0 += 8) {
          double y[8], v[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            y[i] = hcol[min(j0 + i, top)];
            v[i] = Vl[r * NL + min(j0 + i, top)];
          }
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (j0 + i <= top) acc += y[i] * v[i];
        }
        xc_st<X2>(a.x + r0 + r, xc_ld(a.x + r0 + r) + acc);
      }
    } else {
      const int q = gm_opaque(threadIdx.x) >> 6, l = gm_opaque(threadIdx.x) & 63;
      if (RW * q < Rc) {
        double acc[RW];
#pragma unroll
        for (int i = 0; i < RW; ++i) acc[i] = 0.0;
        rows_dot(hcol, top + 1, q, l, acc);
        const double sum = gw_reduce_rows<RW>(acc);
        const int row = RW * q + gw_row<RW>(l);
        if (l < RW && row < Rc) xc_st<X2>(a.x + r0 + row, xc_ld(a.x + r0 + row) + sum);
      }
    }
    if (reason) break;
    if (its >= a.maxit) {
      reason = -2;
      break;
    }
    // every workgroup's rows of x before the next residual; then what is left
    // of the last steps' exchange values is cleared (before the residual's
    // barrier)
    if (!xc_sync<X2>(a.sync, P, c, ++bk, s_err)) break;
    for (int k = 0; k < 3; ++k) coopw_clear<X2>(a, c, r0, Rc, k, min(it, kmax + 1), gm_opaque(threadIdx.x), T);
  }
  // The last workgroup to end its part without a time-out reports the result
  // (all hold the same one).  A workgroup that gives up raises its flag of the
  // last barrier before the error word is looked at, and others may then pass
  // that barrier; it is not counted, so the status stays the time-out that
  // k_coop_prep wrote.
  if (threadIdx.x == 0) {
    if (*s_err) {
      a.s->its = its;
    } else if (__hip_atomic_fetch_add(a.sync + kDoneSlot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u ==
               (unsigned)P) {
      a.s->its = its;
      a.s->reason = reason;
      a.s->rn0 = rn0;
      a.s->ttol = ttol;
      a.s->xmode = X2 ? 1 : 2;
    }
  }
}


// One cooperative solve by the workgroup of rank c (of a.P, all on one XCD
// when the XCD ids they publish at the first barrier agree).
template <int RW, int CQ>
__device__ __forceinline__ void coopw_run(const GmCoopWArgs& a, int c, double* dyn, double* red, double* s_val,
                                          int* s_flag, int* s_err) {
  if (threadIdx.x == 0) {
    *s_err = 0;
    __hip_atomic_store(a.sync + kXccSlot + c, gw_xcc_id() + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  for (int k = 0; k < 3; ++k)
    coopw_clear<false>(a, c, c * a.R, min(a.nf, (c + 1) * a.R) - c * a.R, k, a.kmax + 1, threadIdx.x, kGmT);
  // barrier 1 at device scope; then every workgroup reads the P XCD ids
  // (the same values, so the same decision everywhere)
  if (xc_sync<false>(a.sync, a.P, c, 1u, s_err)) {
    if (threadIdx.x < 64) {
      const int lane = threadIdx.x;
      const unsigned v = lane < a.P ? xc_ldu(a.sync + kXccSlot + lane) : 0u;
      const unsigned v0 = __builtin_amdgcn_readfirstlane(v);
      const bool same = a.l2x && __all(lane >= a.P || v == v0);
      if (lane == 0) s_flag[0] = same;
    }
    __syncthreads();
    if (s_flag[0]) coopw_solve<RW, CQ, true>(a, c, 1u, dyn, red, s_val, s_flag, s_err);
    else coopw_solve<RW, CQ, false>(a, c, 1u, dyn, red, s_val, s_flag, s_err);
  }
}

// One solve, or up to kCoopMulti solves in one launch, solve k on XCD a[k].xcd
// (P workgroups per XCD are launched): the workgroups on that XCD (XCC_ID)
// claim its ranks in turn, those on XCDs no solve names, or past a solve's P,
// leave at once.  Every XCD's workgroups belong to this launch, so no solve
// waits for CUs another solve holds.  A single solve with xcd < 0 takes
// workgroups 0, 8, 16, ... (one XCD when the dispatcher starts the launch's
// round on it).
constexpr int kCoopMulti = 8;
struct GmCoopWMulti {
  int n;
  GmCoopWArgs a[kCoopMulti];
};

template <int RW, int CQ>
__global__ void __launch_bounds__(kGmT) k_gmres_coopw(GmCoopWMulti m) {
  __shared__ int s_c, s_k;
  if (threadIdx.x == 0) {
    int k = -1, c = -1;
    if (m.a[0].xcd < 0) {
      k = 0;
      if (blockIdx.x % 8 == 0) c = (int)(blockIdx.x / 8);
    } else {
      const int id = (int)gw_xcc_id();
      for (int j = 0; j < m.n; ++j)
        if (m.a[j].xcd == id) k = j;
      if (k >= 0)
        c = (int)__hip_atomic_fetch_add(m.a[k].sync + kClaimSlot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_c = k >= 0 && c < m.a[k].P ? c : -1;
    s_k = k;
  }
  __syncthreads();
  const int c = s_c;
  if (c < 0) return;
  const int k = __builtin_amdgcn_readfirstlane(s_k);
  extern __shared__ double dyn[];
  __shared__ double red[kGmT / 64];
  __shared__ double s_val[2];
  __shared__ int s_flag[3];
  __shared__ int s_err;
  coopw_run<RW, CQ>(m.a[k], c, dyn, red, s_val, s_flag, &s_err);
}

// before a cooperative launch: the barrier blocks of its solves cleared and
// their statuses set to reason -3, which stays if no workgroup takes part (one
// workgroup per solve)
__global__ void k_coop_prep(GmCoopWMulti m) {
  const GmCoopWArgs& a = m.a[blockIdx.x];
  if (threadIdx.x < 2 * kCoopSyncDoubles) a.sync[threadIdx.x] = 0u;
  if (threadIdx.x == 0) {
    a.s->reason = -3;
    a.s->its = 0;
  }
}

// dynamic LDS of k_gmres_coopw without the basis (doubles): wl 64, nrm 32,
// hcol/alpha kmax+2 each, grs kmax+1, stg kCwBlk kCwLd, ub nf, and lss kmax in
// the small form (rw = 4)
static size_t coopw_lds_fixed(int rw, int nf, int kmax) {
  return 96 + (size_t)(rw == 4 ? 4 : 3) * kmax + 5 + (size_t)kCwBlk * kCwLd + (size_t)nf;
}

// The small form's split (nf <= 256, four rows per wavefront, the whole basis
// in LDS): the fewest workgroups that hold it.
constexpr int kCoopSmallQ = 4;

bool gmres_coop_plan(int nf, int kmax, size_t max_lds, int* P, int* R) {
  static const int cand[] = {2, 4, 8, 16, 32};
  if (nf > 64 * kCoopSmallQ) return false;
  for (int p : cand) {
    const int r = (nf + p - 1) / p;
    if (r < 1 || r > 4 * (kGmT / 64) || (p - 1) * r >= nf) continue;
    if (kGmT / (kmax + 1) < 1) continue;
    if (sizeof(double) * (coopw_lds_fixed(4, nf, kmax) + (size_t)(kmax + 1) * r) + 1024 > max_lds) continue;
    *P = p;
    *R = r;
    return true;
  }
  return false;
}

bool gmres_coopw_plan(int nf, int kmax, size_t max_lds, int ncu, int* P, int* R, int* NL) {
  static const int cand[] = {8, 16, 32};
  if (nf < 2 || nf > 64 * 16 || kmax < 1 || kmax + 1 > kGmT) return false;
  const size_t budget = max_lds > 2048 ? (max_lds - 2048) / sizeof(double) : 0;
  const size_t fixed = coopw_lds_fixed(2, nf, kmax);
  if (fixed >= budget) return false;
  for (int p : cand) {
    if (8 * p > ncu) continue;
    const int r = (nf + p - 1) / p;
    if (r > 2 * (kGmT / 64)) continue;
    const long nl = std::min<long>(kmax + 1, (long)((budget - fixed) / r));
    if (nl < std::min(kmax + 1, 64)) continue;
    *P = (nf + r - 1) / r;  // every workgroup has rows
    *R = r;
    *NL = (int)nl;
    return true;
  }
  return false;
}

static int coopw_lpg(int P) {
  int l = 0;
  while ((1 << l) < P) ++l;
  return l;
}

// Workspace (doubles), laid out by coopw_args.
size_t gmres_coopw_ws(int nf, int kmax, int P, int R, int NL) {
  return kCoopSyncDoubles + ((size_t)3 * (kmax + 1) << coopw_lpg(P)) + (size_t)4 * (kmax + 1) + (size_t)4 * nf +
         (size_t)2 * P + (size_t)(kmax + 1) * kmax + (size_t)3 * kmax + (size_t)P * R * (size_t)std::max(0, kmax + 1 - NL);
}

size_t gmres_coop_ws(int nf, int kmax, int P) { return gmres_coopw_ws(nf, kmax, P, 0, kmax + 1); }

// the kernel arguments of one solve, its workspace laid out in ws
static GmCoopWArgs coopw_args(int nf, int kmax, int maxit, int P, int R, int NL, const double* S, const double* b,
                              double* x, GmresDev* s, double rtol, double atol, double* ws, int xcd) {
  GmCoopWArgs a{};
  a.nf = nf; a.kmax = kmax; a.maxit = maxit; a.P = P; a.lPg = coopw_lpg(P); a.R = R; a.NL = NL; a.xcd = xcd;
  a.S = S; a.b = b; a.x = x; a.s = s; a.rtol = rtol; a.atol = atol;
  a.sync = reinterpret_cast<unsigned*>(ws);
  a.x1 = ws + kCoopSyncDoubles;
  a.x2 = a.x1 + ((size_t)3 * (kmax + 1) << a.lPg);
  a.x3 = a.x2 + (size_t)3 * (kmax + 1);
  a.rfull = a.x3 + (size_t)3 * nf;
  a.norms = a.rfull + nf;
  a.yg = a.norms + (size_t)2 * P;
  a.Ht = a.yg + (kmax + 1);
  a.rot = a.Ht + (size_t)(kmax + 1) * kmax;
  a.Vg = a.rot + (size_t)3 * kmax;
  // IB_GMRES_L2_EXCHANGE=0 keeps the device-scope exchange even when every
  // workgroup is on one XCD (the results are the same bits either way)
  const char* e = std::getenv("IB_GMRES_L2_EXCHANGE");
  a.l2x = e && std::atoi(e) == 0 ? 0 : 1;
  // IB_GMRES_FAIL_RANK=c lets workgroup c time out at the end of a cycle (the
  // tests' way to that path)
  const char* f = std::getenv("IB_GMRES_FAIL_RANK");
  a.fail_rank = f ? std::atoi(f) : -1;
  return a;
}

// register columns per lane of the kernel instance for nf
static int coopw_cq(int nf) { return nf <= 64 * 8 ? 8 : nf <= 64 * 13 ? 13 : 16; }

static const void* coopw_kernel(int rw, int cq) {
  if (rw == 4) return (const void*)k_gmres_coopw<4, kCoopSmallQ>;
  return cq == 8 ? (const void*)k_gmres_coopw<2, 8>
                 : cq == 13 ? (const void*)k_gmres_coopw<2, 13> : (const void*)k_gmres_coopw<2, 16>;
}

// the solves of m (one register layout) in one launch, P workgroups per XCD.
// An ordinary launch: the barriers are the kernel's own (no runtime grid
// synchronisation resources), one workgroup per CU; a workgroup that is not
// resident in time makes the others leave with reason -3 instead of waiting
// for ever.
static void coopw_launch(hipStream_t st, int rw, const GmCoopWMulti& m, int nxcd) {
  size_t lds = 0;
  int maxP = 0;
  for (int k = 0; k < m.n; ++k) {
    const GmCoopWArgs& a = m.a[k];
    lds = std::max(lds, sizeof(double) * (coopw_lds_fixed(rw, a.nf, a.kmax) + (size_t)a.R * a.NL));
    maxP = std::max(maxP, a.P);
  }
  // barrier words cleared by a kernel (a memset node misbehaves on graph replays)
  hipLaunchKernelGGL(k_coop_prep, dim3(m.n), dim3(2 * kCoopSyncDoubles), 0, st, m);
  IB_LAUNCH_CHECK();
  const int nwg = (m.a[0].xcd < 0 ? 8 : std::max(nxcd, 1)) * maxP;
  void* args[] = {(void*)&m};
  IB_HIP(hipLaunchKernel(coopw_kernel(rw, coopw_cq(m.a[0].nf)), dim3(nwg), dim3(kGmT), args, lds, st));
  IB_LAUNCH_CHECK();
}

void gmres_coop(hipStream_t st, int nf, int kmax, int maxit, int P, int R, const double* S, const double* b, double* x,
                GmresDev* s, double rtol, double atol, double* ws, int xcd, int nxcd) {
  GmCoopWMulti m{};
  m.n = 1;
  m.a[0] = coopw_args(nf, kmax, maxit, P, R, kmax + 1, S, b, x, s, rtol, atol, ws, xcd);
  coopw_launch(st, 4, m, nxcd);
}

void gmres_coopw(hipStream_t st, int nf, int kmax, int maxit, int P, int R, int NL, const double* S, const double* b,
                 double* x, GmresDev* s, double rtol, double atol, double* ws, int xcd, int nxcd) {
  GmCoopWMulti m{};
  m.n = 1;
  m.a[0] = coopw_args(nf, kmax, maxit, P, R, NL, S, b, x, s, rtol, atol, ws, xcd);
  coopw_launch(st, 2, m, nxcd);
}

bool gmres_coopw_multi_ok(int nf_a, int nf_b) { return coopw_cq(nf_a) == coopw_cq(nf_b); }

void gmres_coopw_multi(hipStream_t st, int n, const CoopWJob* jobs, const int* xcds, int nxcd) {
  if (n < 1 || n > kCoopMulti || n > std::max(nxcd, 1))
    throw HipError("gmres_coopw_multi: between 1 and min(8, XCDs) solves per launch");
  GmCoopWMulti m{};
  m.n = n;
  for (int k = 0; k < n; ++k) {
    const CoopWJob& j = jobs[k];
    if (coopw_cq(j.nf) != coopw_cq(jobs[0].nf)) throw HipError("gmres_coopw_multi: solves of different register layouts");
    m.a[k] = coopw_args(j.nf, j.kmax, j.maxit, j.P, j.R, j.NL, j.S, j.b, j.x, j.s, j.rtol, j.atol, j.ws, xcds[k]);
  }
  coopw_launch(st, 2, m, nxcd);
}

// the kernel also has a few hundred bytes of static shared memory, so its
// dynamic share stops 1 KiB short of the device limit (as gmres_dense assumes)
void gmres_dense_set_max_lds(size_t bytes) {
  if (bytes <= 1024) return;
  IB_HIP(hipFuncSetAttribute((const void*)k_gmres_dense<24>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)(bytes - 1024)));
  const void* coop[] = {coopw_kernel(4, 0),
                        coopw_kernel(2, 8),
                        coopw_kernel(2, 13),
                        coopw_kernel(2, 16)};
  for (const void* f : coop)
    IB_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(bytes - 1024)));
}

// ------------------------------------------------------------------------
// Dense Cholesky for the numerically stationary path (num_stat): A = U^T U
// from the upper triangle of a column-major n x n matrix, in place, and the
// explicit inverse A^-1 = U^-1 U^-T, so that each step's solve is one
// matrix-vector product.
// ------------------------------------------------------------------------

// row k of U: U(k,k) = sqrt(A(k,k)), U(k,j) = A(k,j) / U(k,k) for j > k
__global__ void __launch_bounds__(256) k_chol_pivot(int n, double* __restrict__ A, int k, int* __restrict__ err) {
  const double d = A[(long)k * n + k];
  const double dk = d > 0.0 ? sqrt(d) : 1.0;
  if (threadIdx.x == 0 && !(d > 0.0)) err[0] = 1;
  for (int j = k + 1 + threadIdx.x; j < n; j += blockDim.x) A[(long)j * n + k] = A[(long)j * n + k] / dk;
  __syncthreads();
  if (threadIdx.x == 0) A[(long)k * n + k] = dk;
}

// trailing update A(i,j) -= U(k,i) U(k,j) for k < i <= j (16 x 16 tiles)
__global__ void __launch_bounds__(256) k_chol_update(int n, double* __restrict__ A, int k) {
  const int i = k + 1 + blockIdx.x * 16 + threadIdx.x % 16;
  const int j = k + 1 + blockIdx.y * 16 + threadIdx.x / 16;
  if (i >= n || j >= n || i > j) return;
  A[(long)j * n + i] = A[(long)j * n + i] - A[(long)i * n + k] * A[(long)j * n + k];
}

// column c of A^-1: U^T y = e_c (forward), U x = y (backward); one workgroup per column
__global__ void __launch_bounds__(256) k_chol_inverse(int n, const double* __restrict__ U, double* __restrict__ Ainv) {
  extern __shared__ double y[];
  const int c = blockIdx.x;
  for (int j = threadIdx.x; j < n; j += blockDim.x) y[j] = j == c ? 1.0 : 0.0;
  __syncthreads();
  for (int i = c; i < n; ++i) {
    const double yi = y[i] / U[(long)i * n + i];
    __syncthreads();
    for (int j = i + 1 + threadIdx.x; j < n; j += blockDim.x) y[j] = y[j] - U[(long)j * n + i] * yi;
    if (threadIdx.x == 0) y[i] = yi;
    __syncthreads();
  }
  for (int i = n - 1; i >= 0; --i) {
    const double xi = y[i] / U[(long)i * n + i];
    __syncthreads();
    for (int j = threadIdx.x; j < i; j += blockDim.x) y[j] = y[j] - U[(long)i * n + j] * xi;
    if (threadIdx.x == 0) y[i] = xi;
    __syncthreads();
  }
  for (int j = threadIdx.x; j < n; j += blockDim.x) Ainv[(long)c * n + j] = y[j];
}

void chol_factor(hipStream_t st, int n, double* A, int* err) {
  for (int k = 0; k < n; ++k) {
    hipLaunchKernelGGL(k_chol_pivot, dim3(1), dim3(256), 0, st, n, A, k, err);
    IB_LAUNCH_CHECK();
    const int m = n - k - 1;
    if (m > 0) {
      hipLaunchKernelGGL(k_chol_update, dim3(ceil_div(m, 16), ceil_div(m, 16)), dim3(256), 0, st, n, A, k);
      IB_LAUNCH_CHECK();
    }
  }
}

void chol_inverse(hipStream_t st, int n, const double* U, double* Ainv, size_t max_lds) {
  const size_t lds = sizeof(double) * (size_t)n;
  if (lds > max_lds) throw HipError("num_stat: Schur matrix too large for the LDS inverse");
  if (lds > 65536) IB_HIP(hipFuncSetAttribute((const void*)k_chol_inverse, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)lds));
  hipLaunchKernelGGL(k_chol_inverse, dim3(n), dim3(256), lds, st, n, U, Ainv);
  IB_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------
// Multi-kernel Arnoldi step for large systems (the matrix-free form and dense
// matrices past the one-workgroup size): orthogonalisation over many
// workgroups, Givens in one wavefront (affine scan), normalisation.
// ------------------------------------------------------------------------

// w -= sum_j h_j v_j on 64 rows per workgroup (16 wavefronts split the j
// range, partials added in wavefront order); partial ||w||^2 per workgroup
__global__ void __launch_bounds__(1024) k_gm_orth(int nf, int kmax, double* __restrict__ V,
                                                  const GmresDev* __restrict__ s, const double* __restrict__ H,
                                                  double* __restrict__ pnorm) {
  __shared__ double part[16][64];
  if (s->reason) return;
  const int it = s->it, ld = kmax + 1;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r = blockIdx.x * 64 + lane;
  const double* h = H + (long)it * ld;
  double* w = V + (long)(it + 1) * nf;
  const int jn = it + 1, per = (jn + 15) / 16;
  const int j0 = min(jn, wv * per), j1 = min(jn, j0 + per);
  double acc = 0.0;
  if (r < nf) {
    for (int j = j0; j < j1; j += 8) {
      double v[8], hv[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int jj = min(j + c, j1 - 1);
        v[c] = V[(long)jj * nf + r];
        hv[c] = h[jj];
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) acc += -(j + c < j1 ? hv[c] : 0.0) * v[c];
    }
  }
  part[wv][lane] = acc;
  __syncthreads();
  if (wv == 0) {
    double pn = 0.0;
    if (r < nf) {
      double a = w[r];
      for (int q = 0; q < 16; ++q) a += part[q][lane];
      w[r] = a;
      pn = a * a;
    }
    pn = gm_wave_sum(pn);
    if (lane == 0) pnorm[blockIdx.x] = pn;
  }
}

// Givens update of the new Hessenberg column (KSPGMRESUpdateHessenberg) by
// wavefront 0: tt from the partial norms (block order), the previous
// rotations as an affine scan, the new rotation, residual estimate and
// stopping tests; advances the status to the next iteration.  Then the
// whole workgroup forms v_(it+1) = w / tt (skipped after a happy breakdown;
// a vector closed at convergence is never used).  Only wavefront 0 reads the
// status: the others take what they need from LDS after the barrier, since
// wavefront 0 rewrites the status while they may not have started.
__global__ void __launch_bounds__(256) k_gm_givens(int kmax, int nf, double* __restrict__ V, GmresDev* s,
                                                   double* __restrict__ H, double* __restrict__ cc,
                                                   double* __restrict__ ss, double* __restrict__ grs,
                                                   const double* __restrict__ pnorm, int nblk) {
  __shared__ double sh_tt;
  __shared__ int sh_go, sh_col;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    if (s->reason) {
      if (lane == 0) sh_go = 0;
    } else {
      const int it = s->it, ld = kmax + 1;
      double* hcol = H + (long)it * ld;
      double a = 0.0;
      for (int b = 0; b < nblk; ++b) a += pnorm[b];
      const double tt = sqrt(a);
      double carry = hcol[0];
      for (int base = 0; base < it; base += 64) {
        const int j = base + lane;
        const bool act = j < it;
        const double c = act ? cc[j] : 1.0, sn = act ? ss[j] : 0.0, hn = act ? hcol[j + 1] : 0.0;
        double A = -sn, B = c * hn;
        gm_affine_scan(A, B);
        const double cnext = A * carry + B;            // carry_(j+1)
        const double cj = gm_shift_up1(cnext, carry);  // carry_j (lane 0: the carry in)
        if (act) hcol[j] = c * cj + sn * hn;
        carry = gm_readlane(cnext, min(63, it - 1 - base));
      }
      if (lane == 0) {
        hcol[it] = carry;
        hcol[it + 1] = tt;
        double hapbnd = fabs(tt / grs[it]);
        if (hapbnd > 1e-30) hapbnd = 1e-30;
        const int hap = tt < hapbnd;
        double res;
        if (!hap) {
          const double t1 = sqrt(hcol[it] * hcol[it] + hcol[it + 1] * hcol[it + 1]);
          const double c = hcol[it] / t1, sn = hcol[it + 1] / t1;
          cc[it] = c;
          ss[it] = sn;
          grs[it + 1] = -sn * grs[it];
          grs[it] = c * grs[it];
          hcol[it] = c * hcol[it] + sn * hcol[it + 1];
          res = fabs(grs[it + 1]);
        } else {
          res = 0.0;
        }
        s->tt = tt;
        s->hap = hap;
        s->it = it + 1;
        s->its = s->its + 1;
        s->res = res;
        int reason = 0;
        if (res <= s->ttol) reason = 1;
        else if (res >= 1e4 * s->rn0) reason = -1;
        if (hap && !reason) reason = 1;
        s->reason = reason;
        sh_go = !reason && !hap;
        sh_col = it + 1;
        sh_tt = tt;
      }
    }
  }
  __syncthreads();
  if (!sh_go) return;
  const double inv = 1.0 / sh_tt;
  double* v = V + (long)sh_col * nf;
  for (int r = threadIdx.x; r < nf; r += blockDim.x) v[r] = v[r] * inv;
}

void gm_start(hipStream_t st, int nf, int kmax, const double* b, const double* Ax, double* V, GmresDev* s, double* H,
              double* grs, double rtol, double atol) {
  (void)kmax;
  (void)H;
  hipLaunchKernelGGL(k_gm_start, dim3(1), dim3(kGmT), 0, st, nf, b, Ax, V, s, grs, rtol, atol);
  IB_LAUNCH_CHECK();
}

void gm_arnoldi(hipStream_t st, int nf, int kmax, double* V, GmresDev* s, double* H, double* cc, double* ss,
                double* grs, double* pnorm) {
  // kmax+1 dot products at most: one wavefront each, 4 per workgroup
  hipLaunchKernelGGL(k_gm_dots, dim3(ceil_div(kmax + 1, 4)), dim3(256), 0, st, nf, kmax, V, s, H);
  IB_LAUNCH_CHECK();
  const int nblk = ceil_div(nf, 64);
  hipLaunchKernelGGL(k_gm_orth, dim3(nblk), dim3(1024), 0, st, nf, kmax, V, s, H, pnorm);
  IB_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_gm_givens, dim3(1), dim3(256), 0, st, kmax, nf, V, s, H, cc, ss, grs, pnorm, nblk);
  IB_LAUNCH_CHECK();
}

void gm_buildsol(hipStream_t st, int nf, int kmax, const double* V, GmresDev* s, const double* H, const double* grs,
                 double* x, double* scratch) {
  const int c = bs_chunk(kmax);
  const size_t lds = sizeof(double) * (size_t)(c + 2) * (kmax + 1);
  hipLaunchKernelGGL(k_gm_buildsol, dim3(1), dim3(kGmT), lds, st, nf, kmax, c, V, s, H, grs, x, scratch);
  IB_LAUNCH_CHECK();
}

}  // namespace ibg
