// rism_kplane64.hip -- the plane pass, lengths along x from 64
#include "rism_kplane.h"

namespace rism {

template bool launch_plane<64, 2>(const PlaneArgs &);
template bool launch_plane<72, 2>(const PlaneArgs &);
template bool launch_plane<80, 2>(const PlaneArgs &);
template bool launch_plane<96, 2>(const PlaneArgs &);

}  // namespace rism
