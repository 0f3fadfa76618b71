// Host build of the rules that choose a kernel (yrtmi_tiles.hpp), for CPU tests.
#include "yrtmi_tiles.hpp"

extern "C" {

int hw_use_bricks(int64_t nx, int64_t ny, int64_t nz, int64_t frames)
{
	return yrtmi::useBricks(nx, ny, nz, frames);
}

}  // extern "C"
