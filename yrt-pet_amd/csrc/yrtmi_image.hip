// Image-space kernels for gfx950: the separable image-space PSF
// (OperatorPsf::convolve, OperatorPsf.cpp:290-375; its device form
// convolve3DSeparable_kernel, ImageSpaceKernels.cu:296-341), and the
// time-averaged moved image.
#include "yrtmi_kernels.hpp"

namespace yrtmi
{

// One output of an axis is sum over i = 0 .. n - 1, ascending, of k[i] *
// in[c + h - i] (circular), each product and sum rounded separately: the
// order of the reference's CPU loop, so the result is bitwise the same.  A
// thread forms M consecutive outputs of a line in registers; per tap it needs
// one new element of the line (get(j): element c + j of the first output's),
// so a voxel costs (M + n - 1) / M reads an axis and two VALU a tap, the taps
// being kernel arguments (uniform: scalar loads).
template <int M, class Get>
__device__ __forceinline__ void convolveLine(const PsfTaps& t, Get&& get, float (&acc)[M])
{
#pragma clang fp contract(off)
	// four taps a round: w[j] = element h - i - 3 + j, moved on by four
	float w[M + 3];
	int e = t.n / 2;  // h - i
#pragma unroll
	for (int j = 0; j < M; j++)
	{
		acc[j] = 0.f;
		w[j + 3] = get(e + j);
	}
	int i = 0;
	for (; i + 4 <= t.n; i += 4, e -= 4)
	{
#pragma unroll
		for (int j = 0; j < 3; j++)
			w[j] = get(e - 3 + j);
#pragma unroll
		for (int u = 0; u < 4; u++)
		{
			const float k = t.k[i + u];
#pragma unroll
			for (int j = 0; j < M; j++)
				acc[j] = acc[j] + k * w[j + 3 - u];
		}
#pragma unroll
		for (int j = M + 2; j >= 4; j--)
			w[j] = w[j - 4];
		// (read only where a tap follows)
		w[3] = (i + 4 < t.n) ? get(e - 4) : 0.f;
	}
	for (; i < t.n; i++, e--)
	{
		const float k = t.k[i];
#pragma unroll
		for (int j = 0; j < M; j++)
			acc[j] = acc[j] + k * w[j + 3];
#pragma unroll
		for (int j = M + 2; j >= 4; j--)
			w[j] = w[j - 1];
		w[3] = (i + 1 < t.n) ? get(e - 1) : 0.f;
	}
}

// x, then y: one workgroup per kPsfTX x TY voxels of a plane (TY 32, or 16
// where kernels of up to 63 taps would take more than 64 KB of LDS), the plane's
// patch with its halo read into LDS once, convolved along x into a second
// LDS array and from there along y.  (Rows are a multiple of 8 plus one word
// apart in both, so the 8 threads of each of 8 rows meet 64 different banks.)
// One pass over memory for two axes; with kPsfZ a PSF of 9 taps of 4 frames
// of 200 x 200 x 128 takes 105 us where three passes, a global load per tap,
// took 460; a copy of the image takes 32.
constexpr int kPsfTX = 64, kPsfM = 8;

__host__ __device__ constexpr int psfPitch(int hx) { return (kPsfTX + 2 * hx + 7) / 8 * 8 + 1; }

__global__ void __launch_bounds__(256) kPsfXY(const float* __restrict__ in,
                                              float* __restrict__ out, PsfTaps tx, PsfTaps ty,
                                              int nx, int ny, int TY, int ty0)
{
	extern __shared__ float sm[];
	const int hx = tx.n / 2, hy = ty.n / 2;
	const int pitch = psfPitch(hx), rows = TY + 2 * hy;
	float* patch = sm;
	float* mid = sm + pitch * rows;  // rows of kPsfTX, kPsfTX + 1 apart
	const int x0 = (int)blockIdx.x * kPsfTX, y0 = (ty0 + (int)blockIdx.y) * TY;
	const int64_t plane = (int64_t)blockIdx.z * nx * ny;
	// util::circular (Tools.cpp:160-167): one wrap (h < n); elements that no
	// output inside the image needs are read somewhere inside it
	auto wrap = [](int q, int n) {
		q = q < 0 ? q + n : (q >= n ? q - n : q);
		return q < n ? q : 0;
	};
	const int lane = (int)(threadIdx.x & 63u),
	          wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	// (a row of at most 64 + 62 elements: two a lane)
	const int xa = wrap(x0 - hx + lane, nx), xb = wrap(x0 - hx + 64 + lane, nx);
	const bool second = lane < 2 * hx;
	// the loads of four rows in flight together
	for (int r0 = wv; r0 < rows; r0 += 16)
	{
		float va[4], vb[4];
#pragma unroll
		for (int j = 0; j < 4; j++)
		{
			const int r = min(r0 + 4 * j, rows - 1);
			const float* line = in + plane + (int64_t)wrap(y0 - hy + r, ny) * nx;
			va[j] = line[xa];
			vb[j] = second ? line[xb] : 0.f;
		}
#pragma unroll
		for (int j = 0; j < 4; j++)
		{
			const int r = r0 + 4 * j;
			if (r < rows)
			{
				patch[r * pitch + lane] = va[j];
				if (second)
					patch[r * pitch + 64 + lane] = vb[j];
			}
		}
	}
	__syncthreads();
	const int c8 = (int)(threadIdx.x & 7u) * kPsfM;
	for (int r = (int)(threadIdx.x >> 3); r < rows; r += 32)
	{
		const float* p = patch + r * pitch + hx + c8;
		float acc[kPsfM];
		convolveLine<kPsfM>(tx, [&](int j) { return p[j]; }, acc);
#pragma unroll
		for (int j = 0; j < kPsfM; j++)
			mid[r * (kPsfTX + 1) + c8 + j] = acc[j];
	}
	__syncthreads();
	const int x = x0 + lane;
	for (int g = wv; g < TY / kPsfM; g += 4)
	{
		const float* p = mid + (hy + g * kPsfM) * (kPsfTX + 1) + lane;
		float acc[kPsfM];
		convolveLine<kPsfM>(ty, [&](int j) { return p[j * (kPsfTX + 1)]; }, acc);
#pragma unroll
		for (int j = 0; j < kPsfM; j++)
		{
			const int y = y0 + g * kPsfM + j;
			if (x < nx && y < ny)
				out[plane + (int64_t)y * nx + x] = acc[j];
		}
	}
}

// z: one thread per column of kPsfMz voxels, x fastest across the threads;
// the columns' overlap is read from cache.
constexpr int kPsfMz = 16;

__global__ void __launch_bounds__(256) kPsfZ(const float* __restrict__ in,
                                             float* __restrict__ out, PsfTaps t, int nxy, int nz,
                                             int tz0)
{
	const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
	if (i >= nxy)
		return;
	const int z0 = (tz0 + (int)blockIdx.y) * kPsfMz;
	const float* p = in + (int64_t)blockIdx.z * nxy * nz + i;
	float acc[kPsfMz];
	convolveLine<kPsfMz>(
	    t,
	    [&](int j) {
		    int q = z0 + j;
		    q = q < 0 ? q + nz : (q >= nz ? q - nz : q);
		    return p[(int64_t)(q < nz ? q : 0) * nxy];
	    },
	    acc);
	float* o = out + (int64_t)blockIdx.z * nxy * nz + i;
#pragma unroll
	for (int j = 0; j < kPsfMz; j++)
		if (z0 + j < nz)
			o[(int64_t)(z0 + j) * nxy] = acc[j];
}

hipError_t launchPsf(const float* in, float* tmp, float* out, const PsfTaps* t, int nx, int ny,
                     int nz, int64_t frames, hipStream_t st)
{
	const int hx = t[0].n / 2, hy = t[1].n / 2;
	auto ldsOf = [&](int TY) {
		return sizeof(float) * (size_t)(psfPitch(hx) + kPsfTX + 1) * (size_t)(TY + 2 * hy);
	};
	const int TY = ldsOf(32) <= 65536 ? 32 : 16;
	const size_t lds = ldsOf(TY);
	const unsigned gx = (unsigned)((nx + kPsfTX - 1) / kPsfTX);
	const int gy = (ny + TY - 1) / TY, gz = (nz + kPsfMz - 1) / kPsfMz;
	const int nxy = nx * ny;
	const unsigned gc = (unsigned)((nxy + 255) / 256);
	// (a grid has at most 65535 tiles, planes and frames on its second and third axes)
	constexpr int64_t kAxis = 65535;
	auto part = [&](int64_t n) { return (unsigned)std::min(kAxis, n); };
	const int64_t planes = frames * nz;
	for (int64_t p = 0; p < planes; p += kAxis)
		for (int y = 0; y < gy; y += (int)kAxis)
			kPsfXY<<<dim3(gx, part(gy - y), part(planes - p)), 256, lds, st>>>(
			    in + p * nxy, tmp + p * nxy, t[0], t[1], nx, ny, TY, y);
	for (int64_t f = 0; f < frames; f += kAxis)
		for (int z = 0; z < gz; z += (int)kAxis)
			kPsfZ<<<dim3(gc, part(gz - z), part(frames - f)), 256, 0, st>>>(
			    tmp + f * nz * nxy, out + f * nz * nxy, t[2], nxy, nz, z);
	return hipGetLastError();
}

// Time-averaged moved image (timeAverageMoveImage_kernel<true>,
// ImageSpaceKernels.cu:191-264, with util::trilinearInterpolateCore,
// ImageUtils.cuh:15-70).  One thread per output voxel, x fastest: the voxel
// centre ((i v - L/2) + off) + v/2 (util::indexToPosition, ImageUtils.cuh:
// 96-101), then per frame in order q = inv * p as nested fmaf (the
// reference kernel's form), c = (q - origin) * (1/v), i0 = floor(c),
// d = c - i0, and the 8 corners in the reference's order, each adding
// fmaf(in[corner] * w_corner, frame_weight, acc) (corners outside the image
// weigh 0 and read voxel 0, as the reference).  The frames are uniform
// across the grid (scalar loads); the gathers of one frame from 64 adjacent
// x voxels touch two or three cache lines per corner row, so the kernel is
// bound by L2 gathers, 32 B of input per frame per voxel from cache and
// 8 B per voxel from HBM.
__global__ void __launch_bounds__(256) kTimeAverageMove(const float* __restrict__ in,
                                                        float* __restrict__ out,
                                                        const float4* __restrict__ frames,
                                                        int n, MoveGeom g)
{
#pragma clang fp contract(off)
	const int total = g.nx * g.ny * g.nz;
	const int stride = (int)(gridDim.x * blockDim.x);
	// the grid coordinate of the interpolation is clamped to [-4, n + 4]:
	// beyond it every corner is outside (weight 0) either way, and the float
	// to int conversion of floor() stays in range
	const float cmax[3] = {(float)g.nx + 4.f, (float)g.ny + 4.f, (float)g.nz + 4.f};
	for (int i = (int)(blockIdx.x * blockDim.x + threadIdx.x); i < total; i += stride)
	{
		const int ix = i % g.nx;
		const int r = i / g.nx;
		const int iy = r % g.ny;
		const int iz = r / g.ny;
		const int id[3] = {ix, iy, iz};
		float p[3];
		for (int a = 0; a < 3; a++)
			p[a] = (((float)id[a] * g.v[a] - 0.5f * g.len[a]) + g.off[a]) + 0.5f * g.v[a];
		float acc = out[i];
		for (int f = 0; f < n; f++)
		{
			const float4 r0 = frames[4 * f], r1 = frames[4 * f + 1], r2 = frames[4 * f + 2];
			const float fw = frames[4 * f + 3].x;
			const float q[3] = {fmaf(r0.x, p[0], fmaf(r0.y, p[1], fmaf(r0.z, p[2], r0.w))),
			                    fmaf(r1.x, p[0], fmaf(r1.y, p[1], fmaf(r1.z, p[2], r1.w))),
			                    fmaf(r2.x, p[0], fmaf(r2.y, p[1], fmaf(r2.z, p[2], r2.w)))};
			int i0[3];
			float d[3];
			for (int a = 0; a < 3; a++)
			{
				const float c = fminf(fmaxf((q[a] - g.origin[a]) * g.inv[a], -4.f), cmax[a]);
				i0[a] = (int)floorf(c);
				d[a] = c - (float)i0[a];
			}
			const bool inx0 = i0[0] >= 0 && i0[0] < g.nx, inx1 = i0[0] + 1 >= 0 && i0[0] + 1 < g.nx;
			const bool iny0 = i0[1] >= 0 && i0[1] < g.ny, iny1 = i0[1] + 1 >= 0 && i0[1] + 1 < g.ny;
			const bool inz0 = i0[2] >= 0 && i0[2] < g.nz, inz1 = i0[2] + 1 >= 0 && i0[2] + 1 < g.nz;
			const int base = i0[0] + i0[1] * g.nx + i0[2] * g.nx * g.ny;
			for (int k = 0; k < 8; k++)
			{
				const int ox = k & 1, oy = (k >> 1) & 1, oz = (k >> 2) & 1;
				const float wx = ox ? d[0] : 1.f - d[0];
				const float wy = oy ? d[1] : 1.f - d[1];
				const float wz = oz ? d[2] : 1.f - d[2];
				const bool ok = (ox ? inx1 : inx0) && (oy ? iny1 : iny0) && (oz ? inz1 : inz0);
				const int idx = ok ? base + ox + oy * g.nx + oz * g.nx * g.ny : 0;
				const float w = ok ? (wx * wy) * wz : 0.f;
				acc = fmaf(in[idx] * w, fw, acc);
			}
		}
		out[i] = acc;
	}
}

hipError_t launchTimeAverageMove(const float* in, float* out, const float4* frames, int n,
                                 const MoveGeom& g, hipStream_t st)
{
	const int64_t total = (int64_t)g.nx * g.ny * g.nz;
	if (total <= 0 || n <= 0)
		return hipSuccess;
	const unsigned grid = (unsigned)std::min<int64_t>((total + 255) / 256, 65536);
	kTimeAverageMove<<<grid, 256, 0, st>>>(in, out, frames, n, g);
	return hipGetLastError();
}

}  // namespace yrtmi
