/* fame_plane32.hip -- FP32 instances of the plane kernels (fame_plane.hpp) */
#include "fame_plane.hpp"

using namespace fame;

hipError_t fame_launch_line32(const KLine& k, int expand, int mode, int nprob, hipStream_t s) { return launch_line<float>(k, expand, mode, nprob, s); }
hipError_t fame_launch_plane32(const KPlane& k, int nprob, hipStream_t s) { return launch_plane<float>(k, nprob, s); }
hipError_t fame_prepare_plane32(int eb, int ec) { return prepare_plane<float>(eb, ec); }
