// rism_kmisc.hip -- FP64 reductions, the AN2 update, initial t, derived fields,
// per-atom and thermodynamic partial sums.
#include <algorithm>

#include "rism_common.h"

namespace rism {

// ---------------------------------------------------------------------------
// FP64 reductions
// ---------------------------------------------------------------------------
// Sums nrow rows of `width` doubles into out[width], for each of
// gridDim.y consecutive blocks of rows (one workgroup per column and block;
// Kahan-compensated per thread, pairwise tree within the workgroup).
__global__ void __launch_bounds__(256)
    k_reduce_cols(const double *__restrict__ in, size_t nrow, int width,
                  double *__restrict__ out, const int *done, const GroupPtrs *grp) {
  __shared__ double sh[256];
  if (grp) {  // grouped launch: this context's partial sums
    const GroupPtrs &g = grp[blockIdx.z];
    done = global_ptr<const int>(g.done);
    in = global_ptr<const double>(g.partial);
    out = global_ptr<double>(g.sums);
  }
  if (done && *done) return;
  const int col = blockIdx.x;
  in += (size_t)blockIdx.y * nrow * width;
  out += (size_t)blockIdx.y * width;
  double a = 0.0, comp = 0.0;  // Kahan-compensated per-thread accumulation
  for (size_t r = threadIdx.x; r < nrow; r += blockDim.x) {
    const double yv = in[r * width + col] - comp;
    const double tv = a + yv;
    comp = (tv - a) - yv;
    a = tv;
  }
  sh[threadIdx.x] = a;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[col] = sh[0];
}

// ---------------------------------------------------------------------------
// AN2 (anderson_cuda.cu:1-22)
// ---------------------------------------------------------------------------
// The reference keeps the slot pairs (T_p, R_p) and forms
//   u = t + s1 (T0 - t) + s2 (T1 - t)
//   v = t + R + s1 (T0 + R0 - t - R) + s2 (T1 + R1 - t - R)
//   t' = u + m (v - u).
// Writing Q = t + m R and P_p = T_p + m R_p this is
//   t' = Q + s1 (P0 - Q) + s2 (P1 - Q),
// so each slot stores P_p (for the update) and R_p (for the Gram matrix), kept
// by pointer rotation.
//
// The residual pass writes Q into the third of three rotating buffers, which
// becomes the new slot's P: the update reads Q, P0, P1 and writes t', 4 words
// per point (k_an2_mix).  Where it did not (no memory for a third buffer, the
// difference-form steps, a t set by the caller) Q is formed here and written
// out, 6 words (k_an2_update).
//
// Picard warm-up (newdt0): t' = t + R, P_b = t + m R.
// Both kernels move two consecutive elements per thread as 16-byte accesses
// (n = natv * N is even: every grid size is even).
// Elementwise kernels move 16 B per lane per field (two FP64 or four FP32
// values).
template <class Re>
struct alignas(16) V16 {
  static constexpr int K = 16 / sizeof(Re);
  Re a[K];
};

// 16-byte non-temporal accesses of the single-use streams of the updates
template <class Re>
struct NTVec;
template <>
struct NTVec<double> {
  typedef double T __attribute__((ext_vector_type(2)));
};
template <>
struct NTVec<float> {
  typedef float T __attribute__((ext_vector_type(4)));
};
template <class Re>
__device__ __forceinline__ V16<Re> ld_nt(const V16<Re> *p) {
  using T = typename NTVec<Re>::T;
  const T v = __builtin_nontemporal_load(reinterpret_cast<const T *>(p));
  V16<Re> r;
#pragma unroll
  for (int k = 0; k < V16<Re>::K; ++k) r.a[k] = v[k];
  return r;
}
template <class Re>
__device__ __forceinline__ void st_nt(V16<Re> *p, const V16<Re> &x) {
  using T = typename NTVec<Re>::T;
  T v;
#pragma unroll
  for (int k = 0; k < V16<Re>::K; ++k) v[k] = x.a[k];
  __builtin_nontemporal_store(v, reinterpret_cast<T *>(p));
}

template <class Re>
__global__ void k_an2_picard(V16<Re> *__restrict__ tnew, const V16<Re> *__restrict__ t,
                             const V16<Re> *__restrict__ R, V16<Re> *__restrict__ Pb, Re mcoef,
                             size_t nv, const int *done, const GroupPtrs *grp) {
  if (grp) {
    const GroupPtrs &g = grp[blockIdx.z];
    done = global_ptr<const int>(g.done);
    tnew = global_ptr<V16<Re>>(g.tnew);
    t = global_ptr<const V16<Re>>(g.t);
    R = global_ptr<const V16<Re>>(g.R);
    Pb = global_ptr<V16<Re>>(g.Pb);
  }
  if (done && *done) return;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  const V16<Re> ti = t[i], ri = R[i];
  V16<Re> a, b;
#pragma unroll
  for (int k = 0; k < V16<Re>::K; ++k) {
    a.a[k] = ti.a[k] + ri.a[k];
    b.a[k] = ti.a[k] + mcoef * ri.a[k];
  }
  tnew[i] = a;
  if (Pb) Pb[i] = b;
}

template <class Re>
__global__ void k_an2_mix(V16<Re> *__restrict__ tnew, const V16<Re> *__restrict__ Q,
                          const V16<Re> *__restrict__ P0, const V16<Re> *__restrict__ P1,
                          const double *__restrict__ scal, size_t nv, const int *done,
                          const GroupPtrs *grp) {
  if (grp) {
    const GroupPtrs &g = grp[blockIdx.z];
    done = global_ptr<const int>(g.done);
    tnew = global_ptr<V16<Re>>(g.tnew);
    Q = global_ptr<const V16<Re>>(g.Q);
    P0 = global_ptr<const V16<Re>>(g.P0);
    P1 = global_ptr<const V16<Re>>(g.P1);
    scal = global_ptr<const double>(g.scal);
  }
  if (done && *done) return;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  const Re s1 = (Re)scal[3], s2 = (Re)scal[4];
  const V16<Re> q = ld_nt(Q + i), p0 = ld_nt(P0 + i), p1 = ld_nt(P1 + i);
  V16<Re> a;
#pragma unroll
  for (int k = 0; k < V16<Re>::K; ++k)
    a.a[k] = q.a[k] + s1 * (p0.a[k] - q.a[k]) + s2 * (p1.a[k] - q.a[k]);
  st_nt(tnew + i, a);
}

// Pb may alias P0 or P1 (the slot being retired); each element is read before
// it is written by the same thread.
template <class Re>
__global__ void k_an2_update(V16<Re> *__restrict__ tnew, const V16<Re> *__restrict__ t,
                             const V16<Re> *__restrict__ R, const V16<Re> *P0,
                             const V16<Re> *P1, V16<Re> *Pb, const double *__restrict__ scal,
                             Re mcoef, size_t nv, const int *done, const GroupPtrs *grp) {
  if (grp) {
    const GroupPtrs &g = grp[blockIdx.z];
    done = global_ptr<const int>(g.done);
    tnew = global_ptr<V16<Re>>(g.tnew);
    t = global_ptr<const V16<Re>>(g.t);
    R = global_ptr<const V16<Re>>(g.R);
    P0 = global_ptr<const V16<Re>>(g.P0);
    P1 = global_ptr<const V16<Re>>(g.P1);
    Pb = global_ptr<V16<Re>>(g.Pb);
    scal = global_ptr<const double>(g.scal);
  }
  if (done && *done) return;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  const Re s1 = (Re)scal[3], s2 = (Re)scal[4];
  const V16<Re> ti = ld_nt(t + i), ri = ld_nt(R + i), p0 = ld_nt(P0 + i), p1 = ld_nt(P1 + i);
  V16<Re> a, q;
#pragma unroll
  for (int k = 0; k < V16<Re>::K; ++k) {
    q.a[k] = ti.a[k] + mcoef * ri.a[k];
    a.a[k] = q.a[k] + s1 * (p0.a[k] - q.a[k]) + s2 * (p1.a[k] - q.a[k]);
  }
  st_nt(tnew + i, a);
  st_nt(Pb + i, q);
}

// End of a step in one workgroup per context: the column sums of the residual
// pass's partial sums, rms (cal_rms.cu:20-24), the convergence / divergence flag
// (iterate.cu:50-57) and the mixing coefficients for the next update.
// in: natv consecutive blocks of nrow rows of W sums.  Up to kOneGroupSums of
// them are read here by one workgroup; more are reduced by k_reduce_cols first
// and arrive as one row per site.  One kernel against the two: 64^3, 2 sites
// (3072 sums) 4.4 against 4.0 + 3.0 us and a launch; 144 x 160 x 128, 4 sites
// (34560) 8.1 against 4.8 + 4.6; 256^3, 4 sites (98304) 19.6 against 9.4 + 4.5.
constexpr size_t kOneGroupSums = 3 << 14;
constexpr int kEndThreads = 1024;

// Sums into sh[v W + k] (v < natv, k < W): a thread keeps one column (of one
// site) and every rp-th row, Kahan-compensated, then a tree over the rows.
__device__ __forceinline__ void column_sums(const double *__restrict__ in, size_t nrow, int W,
                                            int natv, double *sh) {
  const int nt = blockDim.x, cols = natv * W;
  const int rp = max(1, nt / cols);  // rows side by side
  const int t = threadIdx.x, row = t / cols, col = t % cols;
  const bool mine = row < rp;
  double a = 0.0, comp = 0.0;
  if (mine) {
    const double *p = in + ((size_t)(col / W) * nrow) * W + col % W;
    auto add = [&](double x) {
      const double yv = x - comp;
      const double tv = a + yv;
      comp = (tv - a) - yv;
      a = tv;
    };
    size_t r = row;
    for (; r + 3 * rp < nrow; r += 4 * rp) {  // four loads in flight
      const double x0 = p[r * W], x1 = p[(r + rp) * W], x2 = p[(r + 2 * rp) * W],
                   x3 = p[(r + 3 * rp) * W];
      add(x0);
      add(x1);
      add(x2);
      add(x3);
    }
    for (; r < nrow; r += rp) add(p[r * W]);
    sh[t] = a;
  }
  __syncthreads();
  for (int n = rp; n > 1;) {
    const int h = (n + 1) / 2;
    if (mine && row + h < n) sh[t] += sh[t + h * cols];
    n = h;
    __syncthreads();
  }
}

// rms, its history and the flags: done = {state, step, count}
__device__ __forceinline__ void step_record(double ss, int natv, size_t N, double tol,
                                            double *scal, double *rms_hist, int *done) {
  // step number: done[2] counts the finished steps of the run
  int step = 0;
  if (done) {
    step = done[2] + 1;
    done[2] = step;
  }
  const double rms = sqrt(ss / ((double)N * natv));
  scal[0] = rms;
  if (rms_hist) rms_hist[step] = rms;
  if (done) {
    if (!isfinite(rms)) {
      done[0] = 2;
      done[1] = step;
    } else if (rms <= tol) {
      done[0] = 1;
      done[1] = step;
    }
  }
}

// AN2: the two-slot system (cal_theta anderson.cu:81-102 with the rho^-1
// weights, leg()'s Gaussian elimination without pivoting anderson.cu:105-130,
// the mp shift anderson.cu:66-67).
__global__ void __launch_bounds__(kEndThreads)
    k_step_finish(const double *__restrict__ in, size_t nrow, const double *__restrict__ rho,
                  int natv, size_t N, double tol, int mixing, double mp, int binary,
                  double *__restrict__ scal, double *__restrict__ rms_hist,
                  int *__restrict__ done, const GroupPtrs *grp, int reduced) {
  __shared__ double sums[kEndThreads];
  if (grp) {
    const GroupPtrs &g = grp[blockIdx.z];
    in = reduced ? global_ptr<const double>(g.sums) : global_ptr<const double>(g.partial);
    scal = global_ptr<double>(g.scal);
    rms_hist = global_ptr<double>(g.rms_hist);
    done = global_ptr<int>(g.done);
  }
  if (done && done[0]) return;
  column_sums(in, nrow, 6, natv, sums);
  if (threadIdx.x != 0) return;
  double ss = 0.0, cc0 = 0.0, cc1 = 0.0, a0 = 0.0, a1 = 0.0, a3 = 0.0;
  for (int v = 0; v < natv; ++v) {
    const double *s = sums + 6 * v;
    const double ir = 1.0 / rho[v];
    ss += s[0];
    cc0 += s[1] * ir;
    cc1 += s[2] * ir;
    a0 += s[3] * ir;
    a1 += s[4] * ir;
    a3 += s[5] * ir;
  }
  step_record(ss, natv, N, tol, scal, rms_hist, done);
  if (mixing) {
    const double a2 = a1;
    double b1 = a1, b3 = a3, c0 = cc0, c1 = cc1;
    const double p = a0;
    b1 /= p;
    const double r = c0 /= p;
    const double q = a2;
    b3 -= q * b1;
    c1 -= q * r;
    const double x1 = c1 / b3;
    const double x0 = c0 - b1 * x1;
    scal[1] = x0;
    scal[2] = x1;
    scal[3] = x0 + mp * ((binary == 0) ? 0 : 1);
    scal[4] = x1 + mp * ((binary == 0) ? 1 : 0);
  }
}

// ---------------------------------------------------------------------------
// End of one Anderson(m) step on the device (no counterpart in the
// reference): rms and the convergence / divergence flag as k_step_finish;
// the weighted dots of the new residual R (buffer cur) with itself and the
// nh history residuals (buffers rb[0..nh), oldest first) enter the dot matrix
// D[m1][m1]; and, when the next update mixes, the coefficients th of
//   min |R - sum_p th_p (R - R_p)|  over the newest k history entries:
// G th = b with G_pq = <R - R_p, R - R_q>, b_p = <R, R - R_p>, G scaled to a
// unit diagonal, Gaussian elimination with partial pivoting; when a pivot
// falls below 1e-12 (or a diagonal is not positive) the oldest entry is left
// out and the solve repeated.  th (zeros for entries left out) goes to
// xcoef[0..nh).  FP64; W = 1 + RISM_MAX_HIST sums per site.
// The first wave holds the 16 x 16 system in registers, lane l row l & 15 and
// the four columns from 4 (l >> 4), and exchanges through shuffles (one thread
// with its arrays in scratch memory took 101 us at m = 10, this 14).
// ---------------------------------------------------------------------------
struct AndmHist {
  int rb[RISM_MAX_HIST];
  int nh;
};
static_assert(RISM_MAX_HIST == 16, "the wave solve holds 16 rows");

// element q & 3 of the four columns of a lane
__device__ __forceinline__ double pick4(const double (&g)[4], int q) {
  const double a = (q & 1) ? g[1] : g[0], b = (q & 1) ? g[3] : g[2];
  return (q & 2) ? b : a;
}

__global__ void __launch_bounds__(kEndThreads)
    k_andm_finish(const double *__restrict__ in, size_t nrow, const double *__restrict__ rho,
                  int natv, size_t N, double tol, int W, double *__restrict__ D, int m1, int cur,
                  AndmHist H, int mixing, double *__restrict__ xcoef, double *__restrict__ scal,
                  double *__restrict__ rms_hist, int *__restrict__ done) {
  __shared__ double sums[kEndThreads];
  __shared__ double dots[1 + RISM_MAX_HIST];  // of R with itself and the history
  __shared__ int rb[RISM_MAX_HIST];
  if (done && done[0]) return;
  column_sums(in, nrow, W, natv, sums);
  const int lane = threadIdx.x, nh = H.nh;
  if (lane < RISM_MAX_HIST) {
#pragma unroll
    for (int p = 0; p < RISM_MAX_HIST; ++p)
      if (p == lane) rb[p] = H.rb[p];
  }
  if (lane <= RISM_MAX_HIST) {
    // weighted dots, weights 1 / rho_v (anderson.cu:37-39)
    double a = 0.0;
    if (lane <= nh)
      for (int v = 0; v < natv; ++v) a += sums[W * v + lane] / rho[v];
    dots[lane] = a;
  }
  __syncthreads();
  if (lane >= 64) return;
  if (lane == 0) {
    double ss = 0.0;
    for (int v = 0; v < natv; ++v) ss += sums[W * v];
    step_record(ss, natv, N, tol, scal, rms_hist, done);
    D[(size_t)cur * m1 + cur] = dots[0];
  }
  if (lane < nh) {
    D[(size_t)cur * m1 + rb[lane]] = dots[1 + lane];
    D[(size_t)rb[lane] * m1 + cur] = dots[1 + lane];
  }
  if (!mixing || nh == 0) return;
  const int r = lane & 15, h = lane >> 4;
  const double rr = dots[0];
  double th = 0.0;  // the coefficient of entry r
  for (int first = 0; first < nh; ++first) {
    const int k = nh - first;
    const bool in_r = r < k;
    const double dp = in_r ? dots[1 + first + r] : 0.0;
    double g[4], b = rr - dp;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int q = 4 * h + c;
      // dots among older residuals: entries of D that no lane writes here
      g[c] = (in_r && q < k) ? rr - dp - dots[1 + first + q] +
                                   D[(size_t)rb[first + r] * m1 + rb[first + q]]
                             : 0.0;
    }
    const double diag = __shfl(pick4(g, r), r + 16 * (r >> 2), 64);  // G_rr
    if (__any(in_r && !(diag > 0.0))) continue;
    const double sc = in_r ? 1.0 / sqrt(diag) : 0.0;
    b *= sc;
#pragma unroll
    for (int c = 0; c < 4; ++c) g[c] *= sc * __shfl(sc, (4 * h + c) & 15, 64);
    bool ok = true;
    for (int col = 0; col < k; ++col) {
      const int hc = 16 * (col >> 2);  // lanes that hold the column
      const double gc = __shfl(pick4(g, col), r + hc, 64);
      // the largest |G_rc|, r >= col, the first of equal ones
      double best = (r >= col && in_r) ? fabs(gc) : -1.0;
      int piv = r;
      for (int off = 8; off > 0; off >>= 1) {
        const double ob = __shfl_xor(best, off, 64);
        const int op = __shfl_xor(piv, off, 64);
        if (ob > best || (ob == best && op < piv)) {
          best = ob;
          piv = op;
        }
      }
      // (a value that is no number loses every comparison: the first row stays)
      if (best < 1.0e-12) {
        ok = false;
        break;
      }
      const int src = (r == col ? piv : (r == piv ? col : r)) + 16 * h;
#pragma unroll
      for (int c = 0; c < 4; ++c) g[c] = __shfl(g[c], src, 64);
      b = __shfl(b, src, 64);
      const double gs = __shfl(pick4(g, col), r + hc, 64);
      const double pv = __shfl(gs, col, 64);
      const double f = r > col ? gs / pv : 0.0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double top = __shfl(g[c], col + 16 * h, 64);
        if (4 * h + c >= col) g[c] -= f * top;
      }
      const double bt = __shfl(b, col, 64);
      b -= f * bt;
    }
    if (!ok) continue;
    double x = 0.0;
    for (int q = k - 1; q >= 0; --q) {  // back substitution, a column at a time
      const double gq = __shfl(pick4(g, q), r + 16 * (q >> 2), 64);
      const double xq = __shfl(b / gq, q, 64);
      if (r == q) x = xq;
      if (r < q) b -= gq * xq;
    }
    // entry first + p has row p
    const double xs = x * sc;
    th = __shfl(xs, (r - first) & 15, 64);
    if (r < first) th = 0.0;
    break;
  }
  if (lane < nh) xcoef[lane] = th;
}

// ---------------------------------------------------------------------------
// Anderson(m): the AN2 update generalised to nh history slots,
//   t' = Q + sum_p x_p (P_p - Q),  Q = t + beta R,
// with the retired slot's P overwritten by Q.  Pb may alias one of the P_p;
// each element is read before the same thread writes it.
// ---------------------------------------------------------------------------
template <class Re>
__global__ void k_andm_update(V16<Re> *__restrict__ tnew, const V16<Re> *__restrict__ t,
                              const V16<Re> *__restrict__ R, HistUpdateT<Re> H, V16<Re> *Pb,
                              const double *__restrict__ xcoef, Re beta, size_t nv,
                              const int *done) {
  if (done && *done) return;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  const V16<Re> ti = ld_nt(t + i), ri = ld_nt(R + i);
  V16<Re> q, a;
#pragma unroll
  for (int k = 0; k < V16<Re>::K; ++k) a.a[k] = q.a[k] = ti.a[k] + beta * ri.a[k];
#pragma unroll
  for (int h = 0; h < RISM_MAX_HIST; ++h) {
    if (h < H.nh) {
      // Pb may be the oldest P_h: this thread reads element i before it writes it
      const V16<Re> p = ld_nt(global_ptr<const V16<Re>>(H.p[h]) + i);
      const Re x = (Re)xcoef[h];
#pragma unroll
      for (int k = 0; k < V16<Re>::K; ++k) a.a[k] = fma(x, p.a[k] - q.a[k], a.a[k]);
    }
  }
  st_nt(tnew + i, a);
  st_nt(Pb + i, q);
}

// the closure exponent -u + t, formed in FP64 and rounded once
__global__ void k_exponent(const double *__restrict__ t, const double *__restrict__ u, size_t n,
                           float *__restrict__ out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (float)(-u[i] + t[i]);
}

// Moves a field between the FP64 frame and the FP32 frame of a correction
// block, whose values are differences from the base point t0:
// up: out = t0 + d (out may be t0 itself); down: out = x - t0 in FP32.
__global__ void k_rebase_up(double *out, const double *t0, const float *__restrict__ d,
                            size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = t0[i] + (double)d[i];
}
__global__ void k_rebase_down(const double *__restrict__ x, const double *__restrict__ t0,
                              float *__restrict__ out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (float)(x[i] - t0[i]);
}

// conversion between the FP64 and FP32 copies of a field
template <class From, class To>
__global__ void k_convert(const From *__restrict__ in, To *__restrict__ out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (To)in[i];
}

// ---------------------------------------------------------------------------
// per-atom integrals of the converged g (cal_grad.cu:44-90, cal_euv.cu:30-70,
// cal_ad1.cu:40-80, cal_ad2.cu:40-75): for each solute atom u, sums over the
// grid points r with |r - r_u| >= sigma_uv / 2 (sigma_uv lambda / 2 for ad1)
// of g_v(r) times
//   kind 0 (grad):  [24 eps s6 (2 s6 - 1) / r^2 + cc q_u q_v / r^3] (r - r_u)
//   kind 1 (euv):   4 eps s6 (s6 - 1) + cc q_u q_v / r          (per site v)
//   kind 2 (ad1):   24 eps s6 (2 s6 - 1) / lambda
//   kind 3 (ad2):   cc q_u q_v / r
// with s6 = (sigma_uv^2 / r^2)^3, eps = sqrt(eps_u eps_v) in J/mol, cc =
// E_h a_0 N_A; kinds 0, 2, 3 weight each site by rho_v.
// Lanes are grid points and a wave keeps the sums of AT atoms in registers
// (one thread per atom left most of a workgroup idle for a molecule's few
// atoms: 80 x 72 x 96, 40 atoms, 2 sites, grad 1112 us and energies 989, now 97
// and 81).  The
// four waves of a workgroup take AT atoms each and share g, formed once per
// point and staged in LDS; 1/r and its powers serve all sites.  FP64 VALU
// work, about 21 + 9 natv operations a pair.
// ---------------------------------------------------------------------------
constexpr int AS_TILE = 256;   // points staged at a time
constexpr int AS_WAVES = 4;

// atoms of a wave: the per-site sums of kind 1 take natv registers each
template <int KIND, int NVM>
constexpr int as_atoms() {
  return (KIND == 1 && NVM > 4) ? 4 : 8;
}
// values per atom record: x, y, z, then per site the squared cutoff, sigma^6,
// the Lennard-Jones factor of the kind and cc q_u q_v
__host__ __device__ constexpr int as_stride(int natv) { return 3 + 4 * natv; }

template <int KIND, int NVM>
__global__ void __launch_bounds__(64 * AS_WAVES)
    k_atom_sums(const double *__restrict__ t, const double *__restrict__ u, Params P,
                const double *__restrict__ adata, int natu, const double *__restrict__ rho,
                size_t slab, double *__restrict__ partial) {
  constexpr int AT = as_atoms<KIND, NVM>();
  constexpr int W = KIND == 0 ? 3 : (KIND == 1 ? NVM : 1);
  __shared__ double sg[NVM][AS_TILE];
  const int nv = P.natv, st = as_stride(nv);
  const int lane = threadIdx.x & 63;
  const int a0 = __builtin_amdgcn_readfirstlane((blockIdx.x * AS_WAVES + (threadIdx.x >> 6)) * AT);
  double acc[AT][W];
#pragma unroll
  for (int a = 0; a < AT; ++a)
#pragma unroll
    for (int k = 0; k < W; ++k) acc[a][k] = 0.0;
  const size_t N = (size_t)P.nx * P.ny * P.nz;
  const size_t p0 = (size_t)blockIdx.y * slab;
  const size_t p1 = p0 + slab < N ? p0 + slab : N;
  for (size_t q0 = p0; q0 < p1; q0 += AS_TILE) {
    const int nq = (int)((p1 - q0) < (size_t)AS_TILE ? (p1 - q0) : (size_t)AS_TILE);
    __syncthreads();
    // g of every site, weighted; zero past the slab's end
#pragma unroll
    for (int v = 0; v < NVM; ++v) {
      if (v < nv) {
        const int k = threadIdx.x;
        double g = 0.0;
        if (k < nq) {
          const size_t i = (size_t)v * N + q0 + k;
          g = closure_g(P.clos, t[i], u[i]);
          if (KIND != 1) g *= rho[v];
        }
        sg[v][k] = g;
      }
    }
    __syncthreads();
    if (a0 >= natu) continue;
    for (int k = lane; k < AS_TILE; k += 64) {
      // past the end: the last point, whose g is zero
      const size_t i = q0 + (k < nq ? k : nq - 1);
      const int x = (int)(i % P.nx), y = (int)((i / P.nx) % P.ny),
                z = (int)(i / ((size_t)P.nx * P.ny));
      const double px = (double)(x - P.nx / 2) * P.dr[0], py = (double)(y - P.ny / 2) * P.dr[1],
                   pz = (double)(z - P.nz / 2) * P.dr[2];
      double g[NVM];
#pragma unroll
      for (int v = 0; v < NVM; ++v) g[v] = v < nv ? sg[v][k] : 0.0;
#pragma unroll
      for (int a = 0; a < AT; ++a) {
        // (a spare atom repeats the last one; its sums are not written)
        const double *ad = adata + (size_t)(a0 + a < natu ? a0 + a : natu - 1) * st;
        const double dx = px - ad[0], dy = py - ad[1], dz = pz - ad[2];
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double ir = rsq_nr(r2);  // NaN at r = 0: inside every cutoff
        const double ir2 = ir * ir, ir6 = ir2 * ir2 * ir2;
        double f = 0.0;
#pragma unroll
        for (int v = 0; v < NVM; ++v) {
          if (v < nv) {
            const double *as = ad + 3 + 4 * v;
            const double s6 = as[1] * ir6;
            double e;
            if (KIND == 0)
              e = fma(as[2] * ir2 * s6, fma(2.0, s6, -1.0), as[3] * (ir2 * ir));
            else if (KIND == 1)
              e = fma(as[2] * s6, s6 - 1.0, as[3] * ir);
            else if (KIND == 2)
              e = as[2] * s6 * fma(2.0, s6, -1.0);
            else
              e = as[3] * ir;
            // r < sigma / 2 is left out (r = 0 included)
            const bool in = r2 >= as[0];
            if constexpr (KIND == 1)
              acc[a][v] += in ? e * g[v] : 0.0;
            else
              f += in ? e * g[v] : 0.0;
          }
        }
        if constexpr (KIND == 0) {
          acc[a][0] = fma(f, dx, acc[a][0]);
          acc[a][1] = fma(f, dy, acc[a][1]);
          acc[a][2] = fma(f, dz, acc[a][2]);
        } else if constexpr (KIND != 1) {
          acc[a][0] += f;
        }
      }
    }
  }
  if (a0 >= natu) return;
  const int width = KIND == 0 ? 3 : (KIND == 1 ? nv : 1);
#pragma unroll
  for (int a = 0; a < AT; ++a)
#pragma unroll
    for (int k = 0; k < W; ++k) {
      double x = acc[a][k];
      for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
      if (lane == 0 && a0 + a < natu && k < width)
        partial[((size_t)blockIdx.y * natu + a0 + a) * width + k] = x;
    }
}

// t = q_v fr (initialize_tuv.cu:19-23)
__global__ void k_init_t(double *__restrict__ t, const double *__restrict__ fr, Params P,
                         size_t N) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N * P.natv) return;
  const int v = (int)(i / N);
  t[i] = P.qv[v] * fr[i - (size_t)v * N];
}

// g = closure(t, u), h = R + g - 1 (the h of the step that produced R)
template <class Re>
__global__ void k_fields(const Re *__restrict__ t, const Re *__restrict__ u,
                         const Re *__restrict__ R, Params P, size_t n, int which,
                         double *__restrict__ out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double ti = (double)t[i];
  const double g = closure_g(P.clos, ti, (double)u[i]);
  if (which == 1)
    out[i] = g;
  else if (which == 2)
    out[i] = (double)R[i] + g - 1.0;
  else
    out[i] = (double)R[i] + g - 1.0 - ti;
}

// ---------------------------------------------------------------------------
// thermodynamics (cal_exchem.cu:55-155, cal_pmv.cu:27-57): per-block FP64
// sums of SC (closure-matched), HNC, GF integrands and h - t, per site.
// ---------------------------------------------------------------------------
template <class Re>
__global__ void __launch_bounds__(256)
    k_thermo_partial(const Re *__restrict__ t, const Re *__restrict__ th,
                     const Re *__restrict__ u, const Re *__restrict__ R, Params P,
                     size_t N, double *__restrict__ partial) {
  // t: the current t (the integrand's t); th: the t of the step that produced
  // R, from which h = R + g(th, u) - 1 is rebuilt (equal unless the loop
  // stopped at maxstep, after an AN2 update)
  __shared__ double sh[4][256 / 64];
  const int v = blockIdx.y;
  const Re *tv = t + (size_t)v * N, *uv = u + (size_t)v * N, *Rv = R + (size_t)v * N;
  const Re *thv = th + (size_t)v * N;
  double s[4] = {0, 0, 0, 0};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (size_t)gridDim.x * blockDim.x) {
    const double tt = (double)tv[i];
    const double g = closure_g(P.clos, (double)thv[i], (double)uv[i]);
    const double h = (double)Rv[i] + g - 1.0;
    const double ehnc = h * 0.5 * tt - (h - tt);
    const double egf = -(h * 0.5 + 1.0) * (h - tt);
    const double ekh = (h > 0.0) ? egf : ehnc;
    // PSE-n (clos = 10 + n): HNC integrand minus (t*)^(n+1)/(n+1)!, t* = -u + t
    const double epse =
        (P.clos >= 10) ? ehnc - pse_excess(P.clos - 10, (double)thv[i] - (double)uv[i]) : ehnc;
    s[0] += (P.clos == 0) ? ekh : epse;
    s[1] += ehnc;
    s[2] += egf;
    s[3] += h - tt;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    double a = s[k];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    s[k] = a;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0)
    for (int k = 0; k < 4; ++k) sh[k][wv] = s[k];
  __syncthreads();
  if (threadIdx.x < 4) {
    double a = 0.0;
    for (int w = 0; w < (int)(blockDim.x / 64); ++w) a += sh[threadIdx.x][w];
    partial[((size_t)v * gridDim.x + blockIdx.x) * 4 + threadIdx.x] = a;
  }
}

// reference-convention spectrum from a raw one (rism_k_get_fk): F = phi * D,
// phi = -i (-1)^(nx/2 + ny/2 + jx + jy + m)
__global__ void k_apply_phase(cplx *__restrict__ s, Params P) {
  const size_t M = P.nz / 2;
  const size_t n = M * P.ny * P.nx;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int jx = (int)(i % P.nx), jy = (int)((i / P.nx) % P.ny), m = (int)(i / ((size_t)P.nx * P.ny));
  const int sg = ((P.nx / 2 + P.ny / 2 + jx + jy + m) & 1) ? -1 : 1;
  const cplx a = s[i];
  s[i] = mk(sg * a.y, -sg * a.x);  // phi = -i sg
}

// Plain streaming copy of n 16-byte vectors: the reference point for the HBM
// traffic counters and for the achievable copy bandwidth (reads n, writes n).
__global__ void __launch_bounds__(256)
    k_copy_stream(const V16<double> *__restrict__ in, V16<double> *__restrict__ out, size_t nv) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += stride)
    st_nt(out + i, ld_nt(in + i));
}

hipError_t run_copy(const double *in, double *out, size_t n, hipStream_t st) {
  if (n % 2) return hipErrorInvalidValue;
  const size_t nv = n / 2;
  // 256 CUs x 8 workgroups, grid-stride beyond that
  const unsigned blocks = (unsigned)std::min<size_t>(nblk(nv, 256), 2048);
  hipLaunchKernelGGL(k_copy_stream, dim3(blocks), dim3(256), 0, st,
                     (const V16<double> *)in, (V16<double> *)out, nv);
  return hipGetLastError();
}

hipError_t run_reduce_cols(const double *in, size_t nrow, int width, int nsets, double *out,
                           const int *done, hipStream_t st, const GroupPtrs *grp, int ngrp) {
  hipLaunchKernelGGL(k_reduce_cols, dim3(width, nsets, grp ? ngrp : 1), dim3(256), 0, st, in,
                     nrow, width, out, done, grp);
  return hipGetLastError();
}

// threads of the step's end: one row of sums per site needs few
static int end_threads(bool reduced) { return reduced ? 256 : kEndThreads; }

hipError_t run_step_finish(const double *partial, size_t nrow, double *sums, const double *rho,
                           int natv, size_t N, double tol, int mixing, double mp, int binary,
                           double *scal, double *rms_hist, int *done, hipStream_t st,
                           const GroupPtrs *grp, int ngrp) {
  const int cols = 6 * natv;
  const bool reduce = nrow * cols > kOneGroupSums;
  if (cols > kEndThreads) return hipErrorInvalidValue;
  if (reduce) {
    const hipError_t e = run_reduce_cols(partial, nrow, 6, natv, sums, done, st, grp, ngrp);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_step_finish, dim3(1, 1, grp ? ngrp : 1), dim3(end_threads(reduce)), 0, st,
                     reduce ? sums : partial, reduce ? (size_t)1 : nrow, rho, natv, N, tol, mixing,
                     mp, binary, scal, rms_hist, done, grp, (int)reduce);
  return hipGetLastError();
}

template <class Re>
static size_t nvec(size_t n) {
  return n / V16<Re>::K;
}
template <class Re>
hipError_t run_an2_picard(Re *tnew, const Re *t, const Re *R, Re *Pb, double m, size_t n,
                          const int *done, hipStream_t st, const GroupPtrs *grp, int ngrp) {
  if (n % V16<Re>::K) return hipErrorInvalidValue;
  const size_t nv = nvec<Re>(n);
  hipLaunchKernelGGL(k_an2_picard<Re>, dim3(nblk(nv, 256), 1, grp ? ngrp : 1), dim3(256), 0, st,
                     (V16<Re> *)tnew, (const V16<Re> *)t, (const V16<Re> *)R, (V16<Re> *)Pb,
                     (Re)m, nv, done, grp);
  return hipGetLastError();
}

template <class Re>
hipError_t run_an2_mix(Re *tnew, const Re *Q, const Re *P0, const Re *P1, const double *scal,
                       size_t n, const int *done, hipStream_t st, const GroupPtrs *grp, int ngrp) {
  if (n % V16<Re>::K) return hipErrorInvalidValue;
  const size_t nv = nvec<Re>(n);
  hipLaunchKernelGGL(k_an2_mix<Re>, dim3(nblk(nv, 256), 1, grp ? ngrp : 1), dim3(256), 0, st,
                     (V16<Re> *)tnew, (const V16<Re> *)Q, (const V16<Re> *)P0,
                     (const V16<Re> *)P1, scal, nv, done, grp);
  return hipGetLastError();
}

template <class Re>
hipError_t run_an2_update(Re *tnew, const Re *t, const Re *R, const Re *P0, const Re *P1, Re *Pb,
                          const double *scal, double m, size_t n, const int *done,
                          hipStream_t st, const GroupPtrs *grp, int ngrp) {
  if (n % V16<Re>::K) return hipErrorInvalidValue;
  const size_t nv = nvec<Re>(n);
  hipLaunchKernelGGL(k_an2_update<Re>, dim3(nblk(nv, 256), 1, grp ? ngrp : 1), dim3(256), 0, st,
                     (V16<Re> *)tnew, (const V16<Re> *)t, (const V16<Re> *)R,
                     (const V16<Re> *)P0, (const V16<Re> *)P1, (V16<Re> *)Pb, scal, (Re)m, nv,
                     done, grp);
  return hipGetLastError();
}

template <class Re>
hipError_t run_andm_update(Re *tnew, const Re *t, const Re *R, const HistUpdateT<Re> &H, Re *Pb,
                           const double *xcoef, double beta, size_t n, const int *done,
                           hipStream_t st) {
  if ((n % V16<Re>::K) || H.nh < 0 || H.nh > RISM_MAX_HIST) return hipErrorInvalidValue;
  const size_t nv = nvec<Re>(n);
  hipLaunchKernelGGL(k_andm_update<Re>, dim3(nblk(nv, 256)), dim3(256), 0, st, (V16<Re> *)tnew,
                     (const V16<Re> *)t, (const V16<Re> *)R, H, (V16<Re> *)Pb, xcoef, (Re)beta,
                     nv, done);
  return hipGetLastError();
}

hipError_t run_andm_finish(const double *partial, size_t nrow, double *sums, const double *rho,
                           int natv, size_t N, double tol, int width, double *D, int m1, int cur,
                           const int *rb, int nh, int mixing, double *xcoef, double *scal,
                           double *rms_hist, int *done, hipStream_t st) {
  if (nh < 0 || nh > RISM_MAX_HIST || m1 > RISM_MAX_HIST + 1 || width != 1 + RISM_MAX_HIST ||
      natv * width > kEndThreads)
    return hipErrorInvalidValue;
  AndmHist H{};
  H.nh = nh;
  for (int p = 0; p < nh; ++p) H.rb[p] = rb[p];
  const bool reduce = nrow * natv * width > kOneGroupSums;
  if (reduce) {
    const hipError_t e = run_reduce_cols(partial, nrow, width, natv, sums, done, st);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_andm_finish, dim3(1), dim3(end_threads(reduce)), 0, st,
                     reduce ? sums : partial, reduce ? (size_t)1 : nrow, rho, natv, N, tol, width,
                     D, m1, cur, H, mixing, xcoef, scal, rms_hist, done);
  return hipGetLastError();
}

template <class From, class To>
hipError_t run_convert(const From *in, To *out, size_t n, hipStream_t st) {
  hipLaunchKernelGGL((k_convert<From, To>), dim3(nblk(n, 256)), dim3(256), 0, st, in, out, n);
  return hipGetLastError();
}

#define INST(Re)                                                                              \
  template hipError_t run_an2_picard<Re>(Re *, const Re *, const Re *, Re *, double, size_t,  \
                                         const int *, hipStream_t, const GroupPtrs *, int);   \
  template hipError_t run_an2_mix<Re>(Re *, const Re *, const Re *, const Re *,                \
                                      const double *, size_t, const int *, hipStream_t,        \
                                      const GroupPtrs *, int);                                 \
  template hipError_t run_an2_update<Re>(Re *, const Re *, const Re *, const Re *, const Re *, \
                                         Re *, const double *, double, size_t, const int *,   \
                                         hipStream_t, const GroupPtrs *, int);                \
  template hipError_t run_andm_update<Re>(Re *, const Re *, const Re *,                       \
                                          const HistUpdateT<Re> &, Re *, const double *,      \
                                          double, size_t, const int *, hipStream_t);          \
  template hipError_t run_fields<Re>(const Re *, const Re *, const Re *, const Params &,      \
                                     size_t, int, double *, hipStream_t);                     \
  template hipError_t run_thermo_partial<Re>(const Re *, const Re *, const Re *, const Re *,  \
                                             const Params &, size_t, double *, hipStream_t);
template hipError_t run_convert<double, float>(const double *, float *, size_t, hipStream_t);
hipError_t run_exponent(const double *t, const double *u, size_t n, float *out, hipStream_t st) {
  hipLaunchKernelGGL(k_exponent, dim3(nblk(n, 256)), dim3(256), 0, st, t, u, n, out);
  return hipGetLastError();
}
hipError_t run_rebase_up(double *out, const double *t0, const float *d, size_t n,
                         hipStream_t st) {
  hipLaunchKernelGGL(k_rebase_up, dim3(nblk(n, 256)), dim3(256), 0, st, out, t0, d, n);
  return hipGetLastError();
}
hipError_t run_rebase_down(const double *x, const double *t0, float *out, size_t n,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_rebase_down, dim3(nblk(n, 256)), dim3(256), 0, st, x, t0, out, n);
  return hipGetLastError();
}
template hipError_t run_convert<float, double>(const float *, double *, size_t, hipStream_t);

hipError_t run_init_t(double *t, const double *fr, const Params &P, size_t N, hipStream_t st) {
  hipLaunchKernelGGL(k_init_t, dim3(nblk(N * P.natv, 256)), dim3(256), 0, st, t, fr, P, N);
  return hipGetLastError();
}

template <class Re>
hipError_t run_fields(const Re *t, const Re *u, const Re *R, const Params &P,
                      size_t n, int which, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_fields<Re>, dim3(nblk(n, 256)), dim3(256), 0, st, t, u, R, P, n, which,
                     out);
  return hipGetLastError();
}

int thermo_blocks(size_t N) {
  size_t b = (N + 255) / 256;
  return (int)(b < 1024 ? b : 1024);
}

template <class Re>
hipError_t run_thermo_partial(const Re *t, const Re *th, const Re *u,
                              const Re *R, const Params &P, size_t N, double *partial,
                              hipStream_t st) {
  dim3 grid(thermo_blocks(N), P.natv);
  hipLaunchKernelGGL(k_thermo_partial<Re>, grid, dim3(256), 0, st, t, th, u, R, P, N, partial);
  return hipGetLastError();
}

int atom_sum_stride(int natv) { return as_stride(natv); }

// points per workgroup: whole tiles, at most 1024 slabs
size_t atom_sum_slab(size_t N) {
  size_t s = N / 1024;
  if (s < 1024) s = 1024;
  return (s + AS_TILE - 1) / AS_TILE * AS_TILE;
}

template <int KIND>
static void launch_atom_sums(const double *t, const double *u, const Params &P,
                             const double *adata, int natu, const double *rho, double *partial,
                             hipStream_t st) {
  const size_t N = (size_t)P.nx * P.ny * P.nz, slab = atom_sum_slab(N);
  const unsigned ns = (unsigned)((N + slab - 1) / slab);
  auto go = [&](auto kern, int at) {
    hipLaunchKernelGGL(kern, dim3(nblk(natu, AS_WAVES * at), ns), dim3(64 * AS_WAVES), 0, st, t, u,
                       P, adata, natu, rho, slab, partial);
  };
  if (P.natv <= 2)
    go(k_atom_sums<KIND, 2>, as_atoms<KIND, 2>());
  else if (P.natv <= 4)
    go(k_atom_sums<KIND, 4>, as_atoms<KIND, 4>());
  else
    go(k_atom_sums<KIND, 8>, as_atoms<KIND, 8>());
}

hipError_t run_atom_sums(int kind, const double *t, const double *u, const Params &P,
                         const double *adata, int natu, const double *rho, double *partial,
                         hipStream_t st) {
  if (natu < 1 || P.natv > 8) return hipErrorInvalidValue;
  switch (kind) {
    case 0: launch_atom_sums<0>(t, u, P, adata, natu, rho, partial, st); break;
    case 1: launch_atom_sums<1>(t, u, P, adata, natu, rho, partial, st); break;
    case 2: launch_atom_sums<2>(t, u, P, adata, natu, rho, partial, st); break;
    default: launch_atom_sums<3>(t, u, P, adata, natu, rho, partial, st); break;
  }
  return hipGetLastError();
}

// The twiddle and phase tables of the three axis passes computed on the
// device (the host computes the same values for a context): consecutive
// arrays roots(nx), roots(ny), roots(M), pre(nx), pre(ny), zpre(M),
// zpost(M), M = nz/2, with roots(L)_q = e^{-2 pi i q/L}, pre(n)_j =
// (-1)^j e^{-i pi j/n}, zpre_p = e^{-i pi p/M}, zpost_p = e^{-i pi (2p+1)/nz}.
__global__ void k_fft_tables(int nx, int ny, int nz, cplx *__restrict__ tw) {
  const int M = nz / 2;
  const int total = 2 * nx + 2 * ny + 3 * M;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  int k = i;
  double a;  // angle in units of pi
  double sg = 1.0;
  if (k < nx) {
    a = -2.0 * k / nx;
  } else if ((k -= nx) < ny) {
    a = -2.0 * k / ny;
  } else if ((k -= ny) < M) {
    a = -2.0 * k / M;
  } else if ((k -= M) < nx) {
    a = -(double)k / nx;
    sg = (k & 1) ? -1.0 : 1.0;
  } else if ((k -= nx) < ny) {
    a = -(double)k / ny;
    sg = (k & 1) ? -1.0 : 1.0;
  } else if ((k -= ny) < M) {
    a = -(double)k / M;
  } else {
    k -= M;
    a = -(2.0 * k + 1.0) / nz;
  }
  double sn, cs;
  sincospi(a, &sn, &cs);
  tw[i] = cplx{sg * cs, sg * sn};
}

hipError_t run_fft_tables(int nx, int ny, int nz, cplx *tw, hipStream_t st) {
  const int total = 2 * nx + 2 * ny + 3 * (nz / 2);
  hipLaunchKernelGGL(k_fft_tables, dim3(nblk((size_t)total, 256)), dim3(256), 0, st, nx, ny, nz,
                     tw);
  return hipGetLastError();
}

hipError_t run_apply_phase(cplx *s, const Params &P, hipStream_t st) {
  const size_t n = (size_t)(P.nz / 2) * P.ny * P.nx;
  hipLaunchKernelGGL(k_apply_phase, dim3(nblk(n, 256)), dim3(256), 0, st, s, P);
  return hipGetLastError();
}


INST(double)
INST(float)
#undef INST

}  // namespace rism
