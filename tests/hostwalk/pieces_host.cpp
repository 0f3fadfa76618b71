// Host build of the plan's tile pieces (sidFirst + sidPieces) beside the
// walk they stand for (sidWalk), for CPU tests.
#include "yrtmi_rays.hpp"

#include <vector>

using namespace yrtmi;

namespace
{
struct Piece
{
	float a;
	int x, y, z, segs;
};

template <bool TOF>
bool both(const DImage& P, float3 a, float3 b, const DTof& T, float tofv, const int* l,
          std::vector<Piece>& cut, std::vector<Piece>& walked)
{
	SidRay r;
	if (!sidSetup<TOF, false>(P, a, b, T, tofv, r))
		return false;
	int vx, vy, vz, dx, dy, dz;
	if (sidFirst<false>(P, r, vx, vy, vz, dx, dy, dz))
		sidPieces(P, r, l[0], l[1], l[2], vx, vy, vz, dx, dy, dz,
		          [&](float a0, int x, int y, int z, int segs) {
			          cut.push_back({a0, x, y, z, segs});
		          });
	int last = -1;
	sidWalk<TOF, false>(P, r, T, imageBox(P), true, 0, 0, 0,
	                    [&](int x, int y, int z, uint32_t, float a0, float, uint32_t) {
		                    const int t = ((z >> l[2]) * 1024 + (y >> l[1])) * 1024 + (x >> l[0]);
		                    if (t != last)
			                    walked.push_back({a0, x, y, z, 0});
		                    last = t;
		                    walked.back().segs++;
	                    });
	return true;
}
}  // namespace

extern "C" {

// n rays (p1, p2: n x 3): out[0] rays in the image, [1] pieces of the walks,
// [2] rays whose number of pieces differs, [3] pieces entered at another
// voxel, [4] pieces entered outside the image, [5] pieces whose crossed
// planes are fewer than the walk's segments; *da: the largest difference of
// the entry alphas.
void hw_pieces(const float* imp, int64_t n, const float* p1, const float* p2, int tof,
               const float* tofc, const float* tofv, const int* l, int64_t* out, float* da)
{
	DImage P{};
	P.nx = (int)imp[0];
	P.ny = (int)imp[1];
	P.nz = (int)imp[2];
	P.nt = 1;
	P.vx = imp[3];
	P.vy = imp[4];
	P.vz = imp[5];
	P.lx = imp[6];
	P.ly = imp[7];
	P.lz = imp[8];
	P.fovR = imp[9];
	P.nxy = P.nx * P.ny;
	P.nvox = (int64_t)P.nxy * P.nz;
	const DTof T{tofc[0], tofc[1], tofc[2], rcpNearest(tofc[0])};
	*da = 0.f;
	for (int64_t i = 0; i < n; i++)
	{
		const float3 a = make_float3(p1[3 * i], p1[3 * i + 1], p1[3 * i + 2]),
		             b = make_float3(p2[3 * i], p2[3 * i + 1], p2[3 * i + 2]);
		std::vector<Piece> cut, walked;
		if (!(tof ? both<true>(P, a, b, T, tofv[i], l, cut, walked)
		          : both<false>(P, a, b, T, 0.f, l, cut, walked)))
			continue;
		out[0]++;
		out[1] += (int64_t)walked.size();
		for (const Piece& c : cut)
			out[4] += c.x < 0 || c.x >= P.nx || c.y < 0 || c.y >= P.ny || c.z < 0 || c.z >= P.nz;
		if (cut.size() != walked.size())
		{
			out[2]++;
			continue;
		}
		for (size_t k = 0; k < cut.size(); k++)
		{
			out[3] += cut[k].x != walked[k].x || cut[k].y != walked[k].y || cut[k].z != walked[k].z;
			out[5] += cut[k].segs < walked[k].segs;
			*da = std::max(*da, std::fabs(cut[k].a - walked[k].a));
		}
	}
}

}  // extern "C"
