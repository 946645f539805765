// rism_kplane.h -- passes 2 to 4 of one step in one kernel for small planes:
// DFT along y, DFT along x + OZ + inverse x DFT, inverse y DFT (conventions in
// rism_kxpass.hip).  rism_kplane*.hip instantiate it.
#pragma once
#include "rism_chi.h"

namespace rism {

// One workgroup holds a whole plane m of every site in LDS, reads it once and
// writes it once; the three passes it stands for move it three times.  The
// planes fill the LDS (one workgroup per CU from 64 x 64, 2 sites, on), so a
// stage's LDS accesses, FP64 arithmetic and addresses follow one another: some
// 2 us a stage, four axis transforms of two or three stages (radix 6 saves one
// of 48 points: 14.5 -> 11.5 us at 48^3).  64^3, 2 sites: 16.5 us, about the time
// of the three passes and their launches on one grid; in groups of solutes,
// where the passes are bound by the bytes they move, it gains (48 solutes of 48
// to 96 points a side, half their volume in planes that fit, 48 steps: 63.8 ->
// 61.5 ms).
//
// All butterflies of a stage are shared out over the workgroup, column index
// fastest: lanes of a wave take neighbouring columns, which sit 1 element (y
// stages) or LX + 1 elements (x stages; odd, so that the lanes fall in
// different banks) apart, whatever the stage's stride, and read the same
// twiddle.  A stage reads its inputs into registers, meets a barrier and writes
// its outputs to the same memory.
template <int LX, int LY, int NV>
struct Plane {
  static constexpr int RS = LX + 1;                  // row stride
  static constexpr int SS = LY * RS;                 // site stride
  static constexpr int TAB = 2 * (LX + LY);          // the axes' roots and pre-twiddles
  // registers (complex values) and work (in waves' rounds) of a stage plan
  static constexpr int held(int L, int ncol, int nt) {
    const RadixList rl = make_radices(L, kTens);
    int mx = 0;
    for (int i = 0; i < rl.n; ++i) {
      const int r = rl.r[i], per = (L / r * ncol + nt - 1) / nt;
      mx = per * r > mx ? per * r : mx;
    }
    return mx;
  }
  static constexpr long rounds(int L, int ncol, int nt) {
    const RadixList rl = make_radices(L, kTens);
    long w = 0;
    for (int i = 0; i < rl.n; ++i) {
      const int r = rl.r[i];
      w += (long)((L / r * ncol + nt - 1) / nt) * r * nt;
    }
    return w;
  }
  // threads: the least work done by spare butterflies, among the counts whose
  // stages hold at most 12 complex values a thread (above 768 threads, which have
  // 128 registers) or 18 (168 registers).  Where no count passes (60 x 72 and 60 x
  // 80 either way round, 2 sites; 40 x 60, 4 sites) 1024 threads, which hold the
  // least, 16 (114 to 126 registers, nothing spilled).
  static constexpr int threads() {
    int best = 1024;
    long bw = -1;
    for (int nt = 1024; nt >= 512; nt -= 64) {
      const int hx = held(LX, NV * LY, nt), hy = held(LY, NV * LX, nt);
      if ((hx > hy ? hx : hy) > (nt > 768 ? 12 : 18)) continue;
      const long w = rounds(LX, NV * LY, nt) + rounds(LY, NV * LX, nt);
      if (bw < 0 || w < bw) {
        bw = w;
        best = nt;
      }
    }
    return best;
  }
  static constexpr int NT = threads();
  // the columns of the two axes: element i of column c
  struct X {
    static constexpr int L = LX, NCOL = NV * LY;
    static __device__ __forceinline__ int at(int c, int i) { return c * RS + i; }
  };
  struct Y {
    static constexpr int L = LY, NCOL = NV * LX;
    static __device__ __forceinline__ int at(int c, int i) {
      return (c / LX) * SS + i * RS + c % LX;
    }
  };
};

// The DFT of all columns of axis A.  In reads the first stage's elements, Out
// writes the last stage's; both say (`global`) whether they leave the LDS.
// Ends with a barrier unless Out is global; after loads from global memory it
// meets the one that the tables' writers need.
template <class A, int NT, int S, int STAGE = 0, int NS = 1, class In, class Out>
__device__ __forceinline__ void plane_dft(cplx *lds, const cplx *tw, In &in, Out &out) {
  constexpr RadixList rl = make_radices(A::L, kTens);
  constexpr int R = rl.r[STAGE], NB = A::L / R, TOT = NB * A::NCOL, PER = (TOT + NT - 1) / NT;
  constexpr bool first = STAGE == 0, last = STAGE == rl.n - 1;
  constexpr bool FULL = TOT % NT == 0;
  cplx v[PER][R];
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    // a spare butterfly repeats the last one and stores nothing
    const int i = FULL ? threadIdx.x + b * NT : min((int)threadIdx.x + b * NT, TOT - 1);
    const int c = i % A::NCOL, j = i / A::NCOL;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if constexpr (first)
        v[b][r] = in.get(c, j + r * NB);
      else
        v[b][r] = lds[A::at(c, j + r * NB)];
    }
  }
  if constexpr (first && In::global) __syncthreads();  // the tables
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    const int i = FULL ? threadIdx.x + b * NT : min((int)threadIdx.x + b * NT, TOT - 1);
    const int j = i / A::NCOL;
    if constexpr (first) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[b][r] = in.make(v[b][r], j + r * NB);
    }
    if constexpr (NS > 1) {
      cplx w[R];
      w[1] = tw[(j % NS) * (A::L / (NS * R))];
      twiddle_powers<R>(w);
#pragma unroll
      for (int r = 1; r < R; ++r) v[b][r] = (S < 0) ? cmul(v[b][r], w[r]) : cmulc(v[b][r], w[r]);
    }
    Dft<R, S>::run(v[b]);
  }
  if constexpr (!(first && In::global) && !(last && Out::global)) __syncthreads();
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    const int i = threadIdx.x + b * NT;
    if (FULL || i < TOT) {
      const int c = i % A::NCOL, j = i / A::NCOL;
      const int idx = (j / NS) * NS * R + j % NS;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (last)
          out.put(c, idx + r * NS, v[b][r]);
        else
          lds[A::at(c, idx + r * NS)] = v[b][r];
      }
    }
  }
  if constexpr (!(last && Out::global)) __syncthreads();
  if constexpr (!last) plane_dft<A, NT, S, STAGE + 1, NS * R>(lds, tw, in, out);
}

// LDS to LDS, multiplied by the pre-twiddles (forward) or their conjugates
// (inverse) on the axis where pre is given
template <class A, int S>
struct LdsEnds {
  static constexpr bool global = false;
  cplx *lds;
  const cplx *pre;
  __device__ __forceinline__ cplx get(int c, int i) const { return lds[A::at(c, i)]; }
  __device__ __forceinline__ cplx make(cplx v, int i) const {
    return S < 0 && pre ? cmul(v, pre[i]) : v;
  }
  __device__ __forceinline__ void put(int c, int i, cplx v) const {
    lds[A::at(c, i)] = S > 0 && pre ? cmulc(v, pre[i]) : v;
  }
};
// the spectrum's columns along y
template <int LX, int S>
struct SpecEnds {
  static constexpr bool global = true;
  cplx *plane;      // plane m of site 0
  size_t sstride;   // site stride
  const cplx *pre;
  __device__ __forceinline__ cplx *at(int c, int i) const {
    return plane + (size_t)(c / LX) * sstride + i * LX + c % LX;
  }
  __device__ __forceinline__ cplx get(int c, int i) const {
    const cplx *q = at(c, i);
    return cplx{__builtin_nontemporal_load(&q->x), __builtin_nontemporal_load(&q->y)};
  }
  __device__ __forceinline__ cplx make(cplx v, int i) const { return cmul(v, pre[i]); }
  __device__ __forceinline__ void put(int c, int i, cplx v) const {
    const cplx o = cmulc(v, pre[i]);
    cplx *q = at(c, i);
    __builtin_nontemporal_store(o.x, &q->x);
    __builtin_nontemporal_store(o.y, &q->y);
  }
};

template <int LX, int LY, int NV, int CHI>
__global__ void __launch_bounds__((Plane<LX, LY, NV>::NT))
    k_plane_oz(cplx *__restrict__ spec, const cplx *__restrict__ fkraw, Params P,
               const cplx *__restrict__ twx, const cplx *__restrict__ prex,
               const cplx *__restrict__ twy, const cplx *__restrict__ prey,
               const double *__restrict__ chitab) {
  using PL = Plane<LX, LY, NV>;
  constexpr int NT = PL::NT;
  __shared__ cplx lds[NV * PL::SS];
  __shared__ cplx tab[PL::TAB];
  if (P.grp) {  // grouped launch: this context's spectrum and fk
    const GroupPtrs &g = global_ptr<const GroupPtrs>(P.grp)[blockIdx.z];
    if (stopped(g.done)) return;
    spec = global_ptr<cplx>(g.spec);
    fkraw = global_ptr<const cplx>(g.fk);
  } else if (stopped(P.done)) return;
  const int tid = threadIdx.x, m = blockIdx.x;
  cplx *tx = tab, *ty = tx + LX, *px = ty + LY, *py = px + LX;
  for (int i = tid; i < LX; i += NT) {
    tx[i] = twx[i];
    px[i] = prex[i];
  }
  for (int i = tid; i < LY; i += NT) {
    ty[i] = twy[i];
    py[i] = prey[i];
  }
  cplx *plane = spec + (size_t)m * LY * LX;
  const size_t sstride = (size_t)(P.nz / 2) * LY * LX;

  using X = typename PL::X;
  using Y = typename PL::Y;
  {
    SpecEnds<LX, -1> in{plane, sstride, py};
    LdsEnds<Y, +1> out{lds, nullptr};
    plane_dft<Y, NT, -1>(lds, ty, in, out);
  }
  {
    LdsEnds<X, -1> in{lds, px};
    LdsEnds<X, +1> out{lds, nullptr};
    plane_dft<X, NT, -1>(lds, tx, in, out);
  }
  // OZ: a thread takes the four points (+-kx, +-ky), which share chi (fetching
  // its chi row and fk before the x stages measured the same)
  constexpr int NQ = (LX / 2) * (LY / 2);
  const cplx *fk = fkraw + (size_t)m * LY * LX;
  for (int q = tid; q < NQ; q += NT) {
    const int jx = q % (LX / 2), jy = q / (LX / 2), mx = LX - 1 - jx;
    const auto chi = chi_row<LX, CHI>(chitab, P, NV * NV, jx, jy, m);
    double chr[NV][NV];
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int w = 0; w < NV; ++w) chr[v][w] = chi(v * NV + w);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int y = r ? LY - 1 - jy : jy;
      const int off[2] = {y * PL::RS + jx, y * PL::RS + mx};
      const cplx f[2] = {fk[y * LX + jx], fk[y * LX + mx]};
      oz_points_reg<NV>(lds, PL::SS, off, f, P, chr);
    }
  }
  __syncthreads();
  {
    LdsEnds<X, -1> in{lds, nullptr};
    LdsEnds<X, +1> out{lds, px};
    plane_dft<X, NT, +1>(lds, tx, in, out);
  }
  {
    LdsEnds<Y, -1> in{lds, nullptr};
    SpecEnds<LX, +1> out{plane, sstride, py};
    plane_dft<Y, NT, +1>(lds, ty, in, out);
  }
}

// Which planes the kernel is built for: those that fit the LDS, of the lengths
// that grids of small molecules take.  Every grid of such planes takes it, in
// groups and alone, as a solve must not differ by who shares its launches (the
// passes' radices and so their rounding differ).  Groups decide: 16 solutes of
// 72 x 64 x 32, 2 sites, 205 -> 169 us a step, of 48 x 48 x 32, 4 sites, 183 -> 150.
// Alone, few workgroups (nz / 2) that fill the LDS each leave the chip idle.  A
// step takes 0.86 to 1.02 of the three passes' time for planes of up to 7200
// points of all sites, and of larger ones up to 1.00 from nz = 64 on (from nz = 128
// for 64 x 72, for 48 x 48 with 4 sites, and 1.02 of it for 48 x 96); below, 34.2
// -> 37.3 us at 64 x 64 x 32 and, the most, 40.5 -> 48.3 us at 96 x 48 x 32.
#define RISM_PLANE_LENGTHS(X) X(40) X(48) X(60) X(64) X(72) X(80) X(96)
constexpr bool plane_fits(int nx, int ny, int natv) {
  return 16L * (natv * (long)ny * (nx + 1) + 2 * (nx + ny)) <= 160 * 1024;
}

struct PlaneArgs {
  const Params &P;
  cplx *spec;
  const cplx *fkraw, *twx, *prex, *twy, *prey;
  const double *chitab;
  hipStream_t st;
};

template <int LX, int LY, int NV>
static bool launch_plane_nv(const PlaneArgs &a) {
  if constexpr (plane_fits(LX, LY, NV)) {
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(a.P.nz / 2, 1, a.P.grp ? a.P.ngrp : 1),
                         dim3(Plane<LX, LY, NV>::NT), 0, a.st, a.spec, a.fkraw, a.P, a.twx, a.prex,
                         a.twy, a.prey, a.chitab);
    };
    if (a.P.shell == RISM_CHI_OCTANT) {
      go(k_plane_oz<LX, LY, NV, RISM_CHI_OCTANT>);
      return true;
    }
    if constexpr (LX == LY) {  // the shell table's usual grids
      if (a.P.shell == RISM_CHI_SHELL) {
        go(k_plane_oz<LX, LY, NV, RISM_CHI_SHELL>);
        return true;
      }
    }
  }
  return false;
}
template <int LX, int NV>
bool launch_plane(const PlaneArgs &a) {
  switch (a.P.ny) {
#define X(n) \
  case n:    \
    return launch_plane_nv<LX, n, NV>(a);
    RISM_PLANE_LENGTHS(X)
#undef X
    default:
      return false;
  }
}

}  // namespace rism
