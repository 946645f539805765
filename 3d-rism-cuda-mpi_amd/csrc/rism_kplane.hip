// rism_kplane.hip -- the plane pass, lengths along x up to 60, and its dispatch.
#include "rism_kplane.h"

namespace rism {

#define X(n)                                            \
  extern template bool launch_plane<n, 2>(const PlaneArgs &);
X(64) X(72) X(80) X(96)
#undef X

// whether run_plane takes a step of this grid
bool plane_offered(const Params &P) {
  if ((P.natv != 2 && P.natv != 4) || !plane_fits(P.nx, P.ny, P.natv)) return false;
  if (P.shell != RISM_CHI_OCTANT && !(P.shell == RISM_CHI_SHELL && P.nx == P.ny)) return false;
  auto has = [](int L) {
    switch (L) {
#define X(n) case n:
      RISM_PLANE_LENGTHS(X)
#undef X
      return true;
      default:
        return false;
    }
  };
  return has(P.nx) && has(P.ny);
}

hipError_t run_plane(const Params &P, cplx *spec, const cplx *fkraw, const cplx *twx,
                     const cplx *prex, const cplx *twy, const cplx *prey, const double *chitab,
                     hipStream_t st) {
  const PlaneArgs a{P, spec, fkraw, twx, prex, twy, prey, chitab, st};
  bool ok = false;
  switch (P.nx * 8 + P.natv) {
#define X(n)                       \
  case n * 8 + 2:                  \
    ok = launch_plane<n, 2>(a);    \
    break;
    RISM_PLANE_LENGTHS(X)
#undef X
    case 40 * 8 + 4:
      ok = launch_plane<40, 4>(a);
      break;
    case 48 * 8 + 4:
      ok = launch_plane<48, 4>(a);
      break;
    case 60 * 8 + 4:
      ok = launch_plane<60, 4>(a);
      break;
    default:
      break;
  }
  return ok ? hipGetLastError() : hipErrorInvalidValue;
}

}  // namespace rism
