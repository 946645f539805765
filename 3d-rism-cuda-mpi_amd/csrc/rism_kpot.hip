// rism_kpot.hip -- set-up: the r-space potentials (Lennard-Jones and Coulomb
// sums over the solute's atoms) and the k-space Coulomb term.
#include <algorithm>

#include "rism_common.h"

namespace rism {

// ---------------------------------------------------------------------------
// potentials (cal_LJ.cu:56-81, cal_Coulomb.cu:40-62, cal_potential.cu:39-43)
// ---------------------------------------------------------------------------
// Outputs u[v] = beta sum LJ + q_v de, and fr (first group of sites).
//
// FP64 VALU work, grid points x atoms: what one pair costs decides.
//  * Beyond r = 38 the smoothing 1 - e^{-r} rounds to exactly 1, so de and fr
//    grow by the same q/r, and the reference's two guards (s^2 >= 4e-6 in
//    cal_LJ.cu:11-12, r >= 1e-5 in cal_Coulomb.cu) cannot bind: such a pair
//    needs no exponential and no comparison.  A wave takes these pairs first,
//    then the others, among which only the atoms within the guards' reach of
//    the wave's tile are compared with them.  Which atoms are that far from all
//    of a wave's points is found 64 at a time, one per lane against the wave's
//    tile, and kept as a ballot.
//  * Atoms come sorted by type (equal sigma and epsilon).  4 eps (s^-12 - s^-6)
//    with s^2 = r^2 / sigma^2 is A r^-12 - B r^-6 with A = 4 eps sigma^12 and
//    B = 4 eps sigma^6 the same for all atoms of a type, so a pair adds
//    its r^-6 and r^-12 to two sums, whatever the number of sites, and the
//    sites' A and B enter once per type.  A lane keeps its atom's type, so the
//    runs of a type within 64 atoms are ballots too, and a solute whose atoms
//    are all of different types pays for the A and B of each but not for a
//    test of its own.
//  * A wave owns a compact tile of 16 x 4 x 4 points (four consecutive x per
//    lane), so that the test is sharp, and reads an atom with scalar loads (it
//    is the same for all lanes): no LDS, no barriers.
//  * One kernel for both kinds of pairs, so that u and fr are written once and
//    a tile's atoms are looked at once.  Measured against a kernel for each
//    kind, the second adding to what the first wrote, with a ballot per type:
//    96^3, 4 sites, 6 atoms 65 -> 25 us; 48^3, 8 atoms 20 -> 12 us; 256^3, 4
//    sites, 1500 atoms of few types 19.5 -> 16.2 ms, each of its own type 52 ->
//    26.5 ms.
constexpr int PX = 4;            // consecutive x points of a lane
constexpr int TX = 16, TYZ = 4;  // points of a wave's tile along x, and along y and z
constexpr double kFar = 38.0;    // e^{-r} < 2^-54

// 1/x in FP64 for the rare clamped pairs: the hardware estimate and two
// Newton steps, within an ulp of the IEEE quotient
__device__ __forceinline__ double rcp_nr(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}

// a wave's tile and this lane's points
struct Tile {
  bool ok;
  int x, y, z;
  double rx[PX], ry, rz;
  double cx, cy, cz, rad;  // the tile's centre and the distance of its corners
  __device__ __forceinline__ explicit Tile(const Params &P) {
    const int lane = threadIdx.x & 63;
    const int ntx = (P.nx + TX - 1) / TX, nty = (P.ny + TYZ - 1) / TYZ,
              ntz = (P.nz + TYZ - 1) / TYZ;
    // Workgroups go round-robin to the 8 XCDs, and in the grid's order each XCD
    // would get the same x range of every row when a row takes a divisor of 8
    // of them: with the near pairs in the middle of the box, a few XCDs would
    // do them all.  Each group of 8 is rotated by one more (near pairs of 256^3,
    // 1500 atoms: 7.5 -> 6.9 ms, 300 atoms 1.72 -> 1.56 ms).
    int blk = blockIdx.x;
    if (blk < (int)(gridDim.x & ~7u)) blk = (blk & ~7) | ((blk + (blk >> 3)) & 7);
    const int tile = __builtin_amdgcn_readfirstlane(blk * 4 + (threadIdx.x >> 6));
    ok = tile < ntx * nty * ntz;
    const int x0 = (tile % ntx) * TX, y0 = ((tile / ntx) % nty) * TYZ,
              z0 = (tile / (ntx * nty)) * TYZ;
    x = x0 + PX * (lane & 3);
    y = y0 + ((lane >> 2) & 3);
    z = z0 + (lane >> 4);
    ry = (double)(y - P.ny / 2) * P.dr[1];
    rz = (double)(z - P.nz / 2) * P.dr[2];
#pragma unroll
    for (int p = 0; p < PX; ++p) rx[p] = (double)(x + p - P.nx / 2) * P.dr[0];
    cx = ((double)(x0 - P.nx / 2) + 0.5 * (TX - 1)) * P.dr[0];
    cy = ((double)(y0 - P.ny / 2) + 0.5 * (TYZ - 1)) * P.dr[1];
    cz = ((double)(z0 - P.nz / 2) + 0.5 * (TYZ - 1)) * P.dr[2];
    const double hx = 0.5 * (TX - 1) * P.dr[0], hy = 0.5 * (TYZ - 1) * P.dr[1],
                 hz = 0.5 * (TYZ - 1) * P.dr[2];
    rad = sqrt(hx * hx + hy * hy + hz * hz);
  }
  // whether an atom at p may be within reach of a point of the tile; a
  // coordinate that is no number counts as near
  __device__ __forceinline__ bool near(const double *p, double reach) const {
    const double mx = p[0] - cx, my = p[1] - cy, mz = p[2] - cz;
    const double d2 = fma(mx, mx, fma(my, my, mz * mz)), r = reach + rad;
    return !(d2 >= r * r * (1.0 + 1e-9));
  }
};

// Up to 64 atoms from c0 on, one per lane: its type, and bits of those within
// the smoothing's and the guards' reach of the tile (near) and of the guards
// alone (close).
template <bool COUL>
struct Atoms64 {
  int n, type;
  unsigned long long near, close;
  // atoms: x, y, z, q each, sorted by type; type t has the record
  // tdata[t (1 + 3 natv)]: rc2 = 4e-6 max_v sigma_uv^2, then sigma_uv^2[natv],
  // A[natv], B[natv]
  __device__ __forceinline__ void load(const Tile &T, const double *atoms, const int *types,
                                       const double *tdata, int nv, int natu, int c0) {
    n = natu - c0 < 64 ? natu - c0 : 64;
    const int lane = threadIdx.x & 63, i = c0 + (lane < n ? lane : 0);
    type = types[i];
    const double *p = atoms + 4 * (size_t)i;
    const double guard = sqrt(tdata[(size_t)type * (1 + 3 * nv)]);
    near = __ballot(T.near(p, COUL ? fmax(kFar, guard) : guard)) & all();
    close = __ballot(T.near(p, fmax(1.0e-5, guard))) & near;
  }
  __device__ __forceinline__ unsigned long long all() const {
    return n < 64 ? (1ull << n) - 1 : ~0ull;
  }
  // the type of the first atom of f, and the atoms of f that have it
  __device__ __forceinline__ int run(unsigned long long f, unsigned long long &of) const {
    const int t = __builtin_amdgcn_readlane(type, __builtin_ctzll(f));
    of = f & __ballot(type == t);
    return t;
  }
};

// Up to 4 sites the pair loops fit 128 VGPRs and run four waves per SIMD; more
// would spill at that limit.
template <int G>
constexpr int potential_waves_per_eu() {
  return G <= 4 ? 4 : 1;
}

// 1 - e^{-r} for 0 <= r < 1e4: with k = r 64/ln 2 rounded and f = k ln 2/64 - r,
// |f| <= ln 2 / 128, e^{-r} = t e^f, t = 2^{-(k >> 6)} 2^{-(k & 63)/64} (table
// and polynomial after Tang, ACM TOMS 15, 1989), and the result is formed as
// (1 - t) - t (e^f - 1), so that only t, in the table to half an ulp, and the
// last sum round at its size: e^f - 1 by a polynomial of degree 5 is within
// 4e-17, and k times a one-word ln 2/64 within 3.4e-17 r, 1.3e-17 after the
// factor e^{-r}.  10 operations and a table read against some 23 with the
// library's exponential, whose relative accuracy at large r is lost in 1 -.
__device__ __forceinline__ double one_minus_exp_neg(const double *tab, double r) {
  constexpr double magic = 6755399441055744.0;  // 1.5 2^52: the sum's low word is k
  const double kd = fma(r, 92.332482616893656, magic);
  const int k = (int)(unsigned)__builtin_bit_cast(unsigned long long, kd);
  const double f = fma(kd - magic, 0.010830424696249145, -r);
  double p = fma(f, 1.0 / 120.0, 1.0 / 24.0);
  p = fma(p, f, 1.0 / 6.0);
  p = fma(p, f, 0.5);
  p = fma(p, f, 1.0);
  const double t = ldexp(tab[k & 63], -(k >> 6));
  return fma(-t, p * f, 1.0 - t);
}

template <int G, bool COUL>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(potential_waves_per_eu<G>())))
    k_potential_r(const double *__restrict__ atoms, const int *__restrict__ types,
                  const double *__restrict__ tdata, int natu, int v0, Params P, double ikbt,
                  double ubeta, int write_fr, double *__restrict__ u, double *__restrict__ fr) {
  __shared__ double tab[64];
  if (threadIdx.x < 64) tab[threadIdx.x] = exp2(-(double)threadIdx.x / 64.0);
  __syncthreads();
  const int nv = P.natv;
  const Tile T(P);
  if (!T.ok) return;
  double lj[PX][G], de[PX], ff[PX];
  // sums of r^-6 and r^-12 over atoms of the type cur
  double s6[PX], s12[PX];
  int cur = -1;
#pragma unroll
  for (int p = 0; p < PX; ++p) {
    de[p] = s6[p] = s12[p] = 0.0;
#pragma unroll
    for (int w = 0; w < G; ++w) lj[p][w] = 0.0;
  }
  auto change_type = [&](int t) {
    if (cur >= 0) {
      const double *td = tdata + (size_t)cur * (1 + 3 * nv);
#pragma unroll
      for (int w = 0; w < G; ++w) {
        const double A = td[1 + nv + v0 + w], B = td[1 + 2 * nv + v0 + w];
#pragma unroll
        for (int p = 0; p < PX; ++p) lj[p][w] = fma(A, s12[p], fma(-B, s6[p], lj[p][w]));
      }
#pragma unroll
      for (int p = 0; p < PX; ++p) s6[p] = s12[p] = 0.0;
    }
    cur = t;
  };

  // pairs beyond the smoothing's reach
  auto far = [&](const double *at) {
    const double ax = at[0], aq = at[3];
    const double dy = T.ry - at[1], dz = T.rz - at[2];
    const double dyz = fma(dy, dy, dz * dz);
#pragma unroll
    for (int p = 0; p < PX; ++p) {
      const double dx = T.rx[p] - ax;
      const double ir = rsq_nr(fma(dx, dx, dyz));
      const double ir2 = ir * ir;
      const double ir6 = ir2 * ir2 * ir2;
      s6[p] += ir6;
      s12[p] = fma(ir6, ir6, s12[p]);
      if constexpr (COUL) de[p] = fma(aq, ir, de[p]);
    }
  };
  Atoms64<COUL> A;
  bool any = false;
  for (int c0 = 0; c0 < natu; c0 += 64) {
    A.load(T, atoms, types, tdata, nv, natu, c0);
    const double *at = atoms + 4 * (size_t)c0;
    any |= A.near != 0;
    unsigned long long of;
    for (unsigned long long f = A.all() & ~A.near; f; f &= ~of) {
      const int t = A.run(f, of);
      if (t != cur) change_type(t);
      if (!A.near) {  // consecutive atoms
        const int a1 = 64 - __builtin_clzll(of);
#pragma unroll 2
        for (int a = __builtin_ctzll(of); a < a1; ++a) far(at + 4 * a);
      } else {
        for (unsigned long long b = of; b; b &= b - 1) far(at + 4 * __builtin_ctzll(b));
      }
    }
  }
#pragma unroll
  for (int p = 0; p < PX; ++p) ff[p] = de[p];

  // the others
  constexpr double icut2 = 1.0 / (2.0e-3 * 2.0e-3);  // s^2 >= 4e-6 (cal_LJ.cu:11-12)
  for (int c0 = 0; any && c0 < natu; c0 += 64) {
    if (natu > 64) A.load(T, atoms, types, tdata, nv, natu, c0);
    unsigned long long of;
    for (unsigned long long f = A.near; f; f &= ~of) {
      const int t = A.run(f, of);
      if (t != cur) change_type(t);
      for (unsigned long long b = of & ~A.close; b; b &= b - 1) {
        const double *at = atoms + 4 * (size_t)(c0 + __builtin_ctzll(b));
        const double ax = at[0], aq = at[3];
        const double dy = T.ry - at[1], dz = T.rz - at[2];
        const double dyz = fma(dy, dy, dz * dz);
#pragma unroll
        for (int p = 0; p < PX; ++p) {
          const double dx = T.rx[p] - ax;
          const double r2 = fma(dx, dx, dyz);
          const double ir = rsq_nr(r2);
          const double ir2 = ir * ir;
          const double ir6 = ir2 * ir2 * ir2;
          s6[p] += ir6;
          s12[p] = fma(ir6, ir6, s12[p]);
          if constexpr (COUL) {
            const double qr = aq * ir;
            de[p] += qr;
            ff[p] = fma(qr, one_minus_exp_neg(tab, r2 * ir), ff[p]);
          }
        }
      }
      for (unsigned long long b = of & A.close; b; b &= b - 1) {
        const double *at = atoms + 4 * (size_t)(c0 + __builtin_ctzll(b));
        const double *td = tdata + (size_t)t * (1 + 3 * nv);
        const double ax = at[0], aq = at[3], rc2 = td[0];
        const double dy = T.ry - at[1], dz = T.rz - at[2];
        const double dyz = fma(dy, dy, dz * dz);
#pragma unroll
        for (int p = 0; p < PX; ++p) {
          const double dx = T.rx[p] - ax;
          const double r2 = fma(dx, dx, dyz);
          const double ir = rsq_nr(r2);  // NaN at r2 = 0: both uses below handle it
          const double ir2 = ir * ir;
          if (r2 >= rc2) {
            const double ir6 = ir2 * ir2 * ir2;
            s6[p] += ir6;
            s12[p] = fma(ir6, ir6, s12[p]);
          } else {
#pragma unroll
            for (int w = 0; w < G; ++w) {
              const double sg2 = td[1 + v0 + w];
              const double e4 = td[1 + 2 * nv + v0 + w] * rcp_nr(sg2 * sg2 * sg2);
              const double s2 = fmin(sg2 * ir2, icut2);  // fmin drops the NaN of r = 0
              const double q6 = s2 * s2 * s2;
              lj[p][w] += e4 * q6 * (q6 - 1.0);
            }
          }
          if constexpr (COUL) {
            if (r2 >= 1.0e-10) {  // r >= 1e-5
              const double qr = aq * ir;
              de[p] += qr;
              ff[p] += qr * (1.0 - exp(-(r2 * ir)));
            } else {
              ff[p] += aq;
            }
          }
        }
      }
    }
  }
  change_type(-1);
  if (T.y >= P.ny || T.z >= P.nz) return;
  const size_t N = (size_t)P.nx * P.ny * P.nz;
  const size_t row = ((size_t)T.z * P.ny + T.y) * P.nx + T.x;
#pragma unroll
  for (int p = 0; p < PX; ++p) {
    if (T.x + p >= P.nx) break;
    const double e = de[p] * ubeta;
#pragma unroll
    for (int w = 0; w < G; ++w)
      u[(size_t)(v0 + w) * N + row + p] = lj[p][w] * ikbt + P.qv[v0 + w] * e;
    if (write_fr) fr[row + p] = ff[p] * ubeta;
  }
}

// ---------------------------------------------------------------------------
// fk on the half spectrum (cal_Coulomb.cu:65-79, 90-95), stored raw:
// fkraw = conj(phi(k)) fk, phi(k) = -i (-1)^(nx/2 + ny/2 + jx + jy + m).
// ---------------------------------------------------------------------------
// The sum over atoms of q e^{-i k x} is a matrix product: with
// A[(ky, kz)][u] = q_u e^{-i (ky y_u + kz z_u)} and the real C, S[u][kx] =
// cos, sin(kx x_u), kx > 0, the four real products Re/Im A x C/S give both
// +kx and -kx.  N FMAs per atom (N grid points) on the FP64 matrix cores,
// against a complex rotation and two sums per half-spectrum point in vector
// code.  One wave computes 32 ky x 32 kx of one kz plane: 16 tiles of 16 x 16
// in registers, 5 loads (all from tables of e^{-i k x} per atom and axis, in
// cache) per 16 matrix instructions, no LDS.  The four waves of a workgroup
// take consecutive kz and share the ky and kx tables.
// 512^3, 1500 atoms: 30 -> 14.5 ms (28 TFLOP/s).

// phases of one atom along each axis, cos and sin of k_d x_d (along z times q)
__device__ __forceinline__ cplx phase_x(const Params &P, const double *at, int k) {
  double sn, cs;
  sincos(P.kfac[0] * ((double)k + 0.5) * at[0], &sn, &cs);
  return mk(cs, sn);
}
__device__ __forceinline__ cplx phase_y(const Params &P, const double *at, int jy) {
  double sn, cs;
  sincos(P.kfac[1] * ((double)jy - (double)P.ny / 2.0 + 0.5) * at[1], &sn, &cs);
  return mk(cs, sn);
}
__device__ __forceinline__ cplx phase_z(const Params &P, const double *at, int m) {
  double sn, cs;
  sincos(P.kfac[2] * ((double)m + 0.5) * at[2], &sn, &cs);
  return mk(at[3] * cs, at[3] * sn);
}

// the phases per atom and axis: ex[a][kx > 0], ey[a][ky], ez[a][m], consecutive
// arrays in tab
__global__ void __launch_bounds__(256)
    k_phase_tables(const double *__restrict__ atoms, int na, Params P, cplx *__restrict__ tab) {
  const int nxh = P.nx / 2, M = P.nz / 2, w = nxh + P.ny + M;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)na * w) return;
  const int a = (int)(i / w), k = (int)(i % w);
  const double *at = atoms + 4 * (size_t)a;
  if (k < nxh) {
    tab[(size_t)a * nxh + k] = phase_x(P, at, k);
  } else if (k < nxh + P.ny) {
    tab[(size_t)na * nxh + (size_t)a * P.ny + k - nxh] = phase_y(P, at, k - nxh);
  } else {
    const int m = k - nxh - P.ny;
    tab[(size_t)na * (nxh + P.ny) + (size_t)a * M + m] = phase_z(P, at, m);
  }
}

// Up to this many atoms a workgroup forms its own phases in LDS, 68 an atom,
// and the tables' launch is saved (48^3, 8 atoms 14.1 -> 11.4 us, 16 atoms 16.2
// -> 15.5; 24 atoms would take 19.2 against 18.7).
constexpr int kFkOwn = 16;

typedef double d4 __attribute__((ext_vector_type(4)));

// OWN: atoms' phases formed here, else from the tables
template <bool OWN>
__global__ void __launch_bounds__(256)
    k_fk_half(const double *__restrict__ atoms, const cplx *__restrict__ tab, int na, Params P,
              double ubeta, int add, cplx *__restrict__ fkraw) {
  __shared__ cplx own[OWN ? kFkOwn * 68 : 1];
  const int nxh = P.nx / 2, ny = P.ny, M = P.nz / 2;
  const int nbx = (nxh + 31) / 32, nby = (ny + 31) / 32;
  const int lane = threadIdx.x & 63;
  const int c16 = lane & 15, kq = lane >> 4;
  const int bx = blockIdx.x % nbx, by = (blockIdx.x / nbx) % nby;
  const int m0 = (blockIdx.x / (nbx * nby)) * 4;
  const int mz = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = m0 + mz;
  const int kx0 = bx * 32, ky0 = by * 32;
  if constexpr (OWN) {
    for (int i = threadIdx.x; i < na * 68; i += 256) {
      const int a = i / 68, k = i % 68;
      const double *at = atoms + 4 * (size_t)a;
      own[i] = k < 32 ? phase_x(P, at, kx0 + k)
                      : (k < 64 ? phase_y(P, at, ky0 + k - 32) : phase_z(P, at, m0 + k - 64));
    }
    __syncthreads();
  }
  if (m >= M) return;
  const cplx *ex = tab, *ey = tab + (size_t)na * nxh, *ez = ey + (size_t)na * ny;
  // columns and rows past the end read the last one and are not stored
  int jx[2], jy[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    jx[b] = min(kx0 + 16 * b + c16, nxh - 1);
    jy[b] = min(ky0 + 16 * b + c16, ny - 1);
  }
  // acc[row block][column block]: Ar C, Ai S, Ai C, Ar S
  d4 acc[2][2][4];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[r][c][k] = d4{0, 0, 0, 0};
  struct Op {
    cplx x[2], y[2], z;
  };
  // the operands of atoms k0 .. k0 + 3, one per group of 16 lanes
  auto fetch = [&](int k0) {
    const int a = k0 + kq, ac = min(a, na - 1);
    Op o;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      o.x[b] = OWN ? own[ac * 68 + 16 * b + c16] : ex[(size_t)ac * nxh + jx[b]];
      o.y[b] = OWN ? own[ac * 68 + 32 + 16 * b + c16] : ey[(size_t)ac * ny + jy[b]];
    }
    o.z = OWN ? own[ac * 68 + 64 + mz] : ez[(size_t)ac * M + m];
    if (a >= na) o.z = mk(0.0, 0.0);
    return o;
  };
  Op cur = fetch(0);
  for (int k0 = 0; k0 < na; k0 += 4) {
    const Op nxt = fetch(k0 + 4 < na ? k0 + 4 : k0);  // a step ahead
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      // e^{-i ky y} q e^{-i kz z}
      const double ar = cur.y[r].x * cur.z.x - cur.y[r].y * cur.z.y;
      const double ai = -(cur.y[r].x * cur.z.y + cur.y[r].y * cur.z.x);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        acc[r][c][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, cur.x[c].x, acc[r][c][0], 0, 0, 0);
        acc[r][c][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, cur.x[c].y, acc[r][c][1], 0, 0, 0);
        acc[r][c][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, cur.x[c].x, acc[r][c][2], 0, 0, 0);
        acc[r][c][3] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, cur.x[c].y, acc[r][c][3], 0, 0, 0);
      }
    }
    cur = nxt;
  }
  const double kz = P.kfac[2] * ((double)m + 0.5);
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      // the product's row in element v of a lane
      const int y = ky0 + 16 * r + 4 * v + kq;
      if (y >= ny) continue;
      const double ky = P.kfac[1] * ((double)y - (double)ny / 2.0 + 0.5);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int x = kx0 + 16 * c + c16;
        if (x >= nxh) continue;
        const double kx = P.kfac[0] * ((double)x + 0.5);
        const double rk2 = kx * kx + ky * ky + kz * kz;
        const double f = 4.0 * M_PI * (1.0 / (rk2 * (rk2 + 1.0))) * ubeta;
        const double rc = acc[r][c][0][v], is = acc[r][c][1][v], ic = acc[r][c][2][v],
                     rs = acc[r][c][3][v];
        cplx *row = fkraw + ((size_t)m * ny + y) * P.nx;
#pragma unroll
        for (int s = 0; s < 2; ++s) {  // +kx, -kx
          const int j = s ? nxh - 1 - x : nxh + x;
          const double fre = f * (s ? rc - is : rc + is), fim = f * (s ? ic + rs : ic - rs);
          // conj(phi) = i sg
          const double sg = ((nxh + ny / 2 + y + m + j) & 1) ? -1.0 : 1.0;
          cplx o = mk(-sg * fim, sg * fre);
          if (add) o = o + row[j];
          row[j] = o;
        }
      }
    }
}

hipError_t run_potential_r(const double *atoms, const int *types, const double *tdata, int natu,
                           const Params &P, double ikbt, double ubeta, int do_coul, double *u,
                           double *fr, hipStream_t st) {
  const size_t tiles = (size_t)((P.nx + TX - 1) / TX) * ((P.ny + TYZ - 1) / TYZ) *
                       ((P.nz + TYZ - 1) / TYZ);
  const dim3 grid(nblk(tiles, 4)), block(256);
  for (int v0 = 0; v0 < P.natv; v0 += 8) {
    const int g = min(8, P.natv - v0);
    const int wf = v0 == 0;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, block, 0, st, atoms, types, tdata, natu, v0, P, ikbt, ubeta,
                         wf, u, fr);
    };
    switch (g) {
#define G_CASE(n)                    \
  case n:                            \
    if (do_coul)                     \
      go(k_potential_r<n, true>);    \
    else                             \
      go(k_potential_r<n, false>);   \
    break;
      G_CASE(1) G_CASE(2) G_CASE(3) G_CASE(4) G_CASE(5) G_CASE(6) G_CASE(7) G_CASE(8)
#undef G_CASE
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t run_fk_half(const double *atoms, int natu, const Params &P, double ubeta, cplx *work,
                       size_t nwork, cplx *fkraw, hipStream_t st) {
  // as many atoms at a time as the tables fit the work space
  const size_t per = (size_t)P.nx / 2 + P.ny + P.nz / 2;
  const int chunk = (int)std::min<size_t>((size_t)natu, nwork / per);
  if (chunk < 1) return hipErrorInvalidValue;
  const int nb = ((P.nx / 2 + 31) / 32) * ((P.ny + 31) / 32) * ((P.nz / 2 + 3) / 4);
  if (natu <= kFkOwn) {
    hipLaunchKernelGGL(k_fk_half<true>, dim3(nb), dim3(256), 0, st, atoms, (const cplx *)nullptr,
                       natu, P, ubeta, 0, fkraw);
    return hipGetLastError();
  }
  for (int a0 = 0; a0 < natu; a0 += chunk) {
    const int na = std::min(chunk, natu - a0);
    hipLaunchKernelGGL(k_phase_tables, dim3(nblk(na * per, 256)), dim3(256), 0, st,
                       atoms + 4 * (size_t)a0, na, P, work);
    hipLaunchKernelGGL(k_fk_half<false>, dim3(nb), dim3(256), 0, st, atoms, (const cplx *)work, na,
                       P, ubeta, a0 > 0, fkraw);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace rism
