// Host build of the rules that choose a kernel (yrtmi_tiles.hpp), for CPU tests.
#include "yrtmi_tiles.hpp"

extern "C" {

int hw_use_bricks(int64_t nx, int64_t ny, int64_t nz, int64_t frames, int dd, int rays, int64_t n)
{
	return yrtmi::useBricks(nx, ny, nz, frames, dd != 0, rays, n);
}

// Records per LOR that a DD backprojection without a plan has room for, with
// tiles of 32 x 32 x 8.
int64_t hw_dd_records(int64_t nx, int64_t ny, int64_t nz, float vx, float vy, float vz, float tt,
                      float tz, float ext)
{
	return yrtmi::ddRecordsPerLor(yrtmi::tilesOf(3, nx, ny, nz, 1), vx, vy, vz, tt, tz, ext);
}

}  // extern "C"
