// Tile-binned backprojection (Siddon and distance-driven) for gfx950.
//
// Random FP32 atomics into a 20 MB image run at a few tens of G/s on the
// chip, an order of magnitude below the rate at which rays are walked, so
// the direct backprojection is bound by them.  Here the walk of every
// (LOR, ray) is cut at the boundaries of TX x TY x TZ image tiles:
//
//  plan (once per LOR set; geometry only):
//    kRayPrep     resolve every (LOR, ray) once into the ray table
//    kBin<COUNT>  cut every ray at its tiles (sidPieces), count tile entries
//                 per tile (LDS counters, one global atomic per tile and
//                 workgroup)
//    host         prefix sum -> tile ranges, chunk table
//    kBin<FILL>   cut again, write one record per tile entry into its
//                 tile's range: key = lor * R + ray, the alpha where the
//                 walk enters the tile, the voxel it enters and the ray's
//                 plane shift (sidPlaneShift); a DD record is the LOR alone
//  per backprojection:
//    kTileBack    one workgroup per chunk of a tile's records: re-enter each
//                 ray's walk at its record (sidRestart) or sweep the DD
//                 footprint over the tile, accumulate in the tile held in
//                 LDS, then add the tile to the image with coalesced atomics
//                 (one per touched voxel).
#include "yrtmi_tiles.hpp"

#include <algorithm>
#include <type_traits>

namespace yrtmi
{

__device__ __forceinline__ void ldsAdd(float* p, float v)
{
	__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void ldsAdd64(unsigned long long* p, long long v)
{
	__hip_atomic_fetch_add(p, (unsigned long long)v, __ATOMIC_RELAXED,
	                       __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ int tileOf(const DTiles& T, int f, int vx, int vy,
                                      int vz)
{
	return ((f * T.ntz + (vz >> T.lz)) * T.nty + (vy >> T.ly)) * T.ntx + (vx >> T.lx);
}

// Ray table of a LOR set (rayEntry for every (LOR, ray) t = e * R + r):
// the LOR resolved once (detector pair or histogram bin, LUT, motion,
// frame), the multi-ray line and the image offset.  Skipped LORs get frame -1.
// Distance-driven (DD): the LOR's footprint set-up (ddSetup, ddStore).
// A plane shift beyond the record's range sets *err (the ray is skipped).
template <bool DD, bool TOF, bool S64>
__global__ void __launch_bounds__(256) kRayPrep(KArgs a, float4* __restrict__ tab, int* err)
{
	const int R = a.pr.numRays;
	const int64_t total = lorCount(a) * (int64_t)R;
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride)
	{
		const int64_t e = t / R;
		const int r = (int)(t - e * R);
		const Lor l = fetchLor(a.sc, a.L, lorElement(a, e), a.im.nt);
		if (DD)
		{
			if (l.frame < 0)
			{
				ddStoreSkip(tab, (uint64_t)t);
				continue;
			}
			const float3 d1 = make_float3(l.p1.x - a.im.ox, l.p1.y - a.im.oy, l.p1.z - a.im.oz);
			const float3 d2 = make_float3(l.p2.x - a.im.ox, l.p2.y - a.im.oy, l.p2.z - a.im.oz);
			DDRay D;
			ddSetup<TOF, S64>(a.im, d1, d2, l.n1, l.n2, a.pr, l.tof, false, D);
			ddStore(tab, (uint64_t)t, D, l.frame);
			continue;
		}
		constexpr int V = rayTabVec(S64);
		float3 q1 = make_float3(0.f, 0.f, 0.f), q2 = q1;
		if (l.frame >= 0)
		{
			rayLine(a.pr, l, r, q1, q2);
			q1 = make_float3(q1.x - a.im.ox, q1.y - a.im.oy, q1.z - a.im.oz);
			q2 = make_float3(q2.x - a.im.ox, q2.y - a.im.oy, q2.z - a.im.oz);
		}
		if (S64)
		{
			rayEntry(tab, V, (uint32_t)t, q1, q2, l.frame >= 0 ? l.tof : 0.f,
			         l.frame >= 0 ? l.frame : -1);
			continue;
		}
		// the ray's FP32 set-up and its first voxel
		SidRay sr;
		int vx = 0, vy = 0, vz = 0, dx = 0, dy = 0, dz = 0;
		bool ok = l.frame >= 0 && sidSetup<TOF, false>(a.im, q1, q2, a.pr.tof, l.tof, sr) &&
		          sidFirst<false>(a.im, sr, vx, vy, vz, dx, dy, dz) &&
		          (unsigned)vx < (unsigned)a.im.nx && (unsigned)vy < (unsigned)a.im.ny &&
		          (unsigned)vz < (unsigned)a.im.nz;
		if (ok && (abs(dx) > kMaxShift || abs(dy) > kMaxShift || abs(dz) > kMaxShift))
		{
			atomicOr(err, 2);
			ok = false;
		}
		rayEntry(tab, V, (uint32_t)t, q1, q2,
		         __uint_as_float((uint32_t)vx | ((uint32_t)vy << 10) | ((uint32_t)vz << 20)),
		         (int32_t)(ok ? rayWord(l.frame, dx, dy, dz) : kNoFrame));
		if (ok)
			sidStore(tab + V * (uint64_t)t + 2, sr);
		else
			tab[V * (uint64_t)t + 2] = tab[V * (uint64_t)t + 3] = make_float4(0.f, 0.f, 0.f, 0.f);
	}
}

// The pieces of ray t of the ray table: onRecord(tile, alpha, packed entry,
// segments) for each tile its walk passes through.  FP32 set-up: cut tile by
// tile (sidPieces); FP64: by walking it (its first planes have the set-up's
// own alphas).  A plane shift beyond the record's range sets *err (the ray
// is not binned).
template <bool TOF, bool S64, class Fn>
__device__ __forceinline__ void binRay(const DImage& im, const DTof& tof, const DTiles& T,
                                       const float4* __restrict__ tab, uint32_t t, int* err,
                                       Fn&& onRecord)
{
	constexpr int V = rayTabVec(S64);
	const float4 A = tab[V * (uint64_t)t], Bq = tab[V * (uint64_t)t + 1];
	const float3 q1 = make_float3(A.x, A.y, A.z), q2 = make_float3(A.w, Bq.x, Bq.y);
	SidRay s;
	if constexpr (!S64)
	{
		const float4 s0 = tab[V * (uint64_t)t + 2], s1 = tab[V * (uint64_t)t + 3];
		const uint32_t w = __float_as_uint(Bq.w), fv = __float_as_uint(Bq.z);
		const int frame = (int)(w & 0xffffu);
		if (frame == (int)kNoFrame)
			return;
		sidLoad(q1, q2, s0, s1, s);
		// the entry word's shift bits lie one below the table word's
		const uint32_t sh = (w >> 1) & 0x07ff8000u;
		uint32_t first = 0x80000000u;
		sidPieces(im, s, T.lx, T.ly, T.lz, (int)(fv & 1023u), (int)((fv >> 10) & 1023u),
		          (int)((fv >> 20) & 1023u), (int)((w >> 16) & 15u) - 8,
		          (int)((w >> 20) & 15u) - 8, (int)((w >> 24) & 15u) - 8,
		          [&](float a0, int vx, int vy, int vz, int segs) {
			          onRecord(tileOf(T, frame, vx, vy, vz), a0,
			                   (uint32_t)(vx & (T.tx - 1)) | ((uint32_t)(vy & (T.ty - 1)) << 5) |
			                       ((uint32_t)(vz & (T.tz - 1)) << 10) | sh | first,
			                   segs);
			          first = 0u;
		          });
		return;
	}
	const int frame = __float_as_int(Bq.w);
	if (frame < 0)
		return;
	if (!sidSetup<TOF, S64>(im, q1, q2, tof, Bq.z, s))
		return;
	int dx, dy, dz;
	if (!sidPlaneShift<S64>(im, s, dx, dy, dz))
		return;
	if (abs(dx) > kMaxShift || abs(dy) > kMaxShift || abs(dz) > kMaxShift)
	{
		atomicOr(err, 2);
		return;
	}
	int last = -1, start = 0, nseg = 0;
	float pa = 0.f;
	uint32_t pv = 0;
	sidWalk<TOF, S64>(im, s, tof, imageBox(im), true, 0, 0, 0,
	                  [&](int vx, int vy, int vz, uint32_t, float a0, float, uint32_t) {
		                  const int tl = tileOf(T, frame, vx, vy, vz);
		                  if (tl != last)
		                  {
			                  if (last >= 0)
				                  onRecord(last, pa, pv, nseg - start);
			                  pa = a0;
			                  pv = packEntry(vx & (T.tx - 1), vy & (T.ty - 1), vz & (T.tz - 1),
			                                 dx, dy, dz, last < 0);
			                  start = nseg;
			                  last = tl;
		                  }
		                  nseg++;
	                  });
	if (last >= 0)
		onRecord(last, pa, pv, nseg - start);
}

// DD: the tiles of LOR t's footprint.  The slices of the major axis are
// taken one tile slab at a time, with the footprint ranges of each slice
// (ddSlice, the ranges the sweep itself visits).  Each tile of the bounding
// box of a slab's ranges that some slice reaches gives a record:
// onRecord(tile, 0, first | last << 6, voxels), first and last the slices
// (less the slab's first) that reach it — the sweep of the record goes over
// these slices only — and voxels its number of footprint voxels in the tile.
template <class Fn>
__device__ __forceinline__ void binRayDD(const DImage& im, const DProj& pr, const DTiles& T,
                                         const float4* __restrict__ tab, uint32_t t,
                                         Fn&& onRecord)
{
	const float4* te = tab + kDDVec * (uint64_t)t;
	float4 e[kDDVec];
#pragma unroll
	for (int i = 0; i < kDDVec; i++)
		e[i] = te[i];
	const int frame = ddFrame(e[5]);
	if (frame < 0)
		return;
	DDRay R;
	ddLoad(im, pr, e, false, R);
	const int lm = R.flag_y ? T.ly : T.lx;  // major axis
	const int ln = R.flag_y ? T.lx : T.ly;  // minor axis
	for (int s0 = R.xy_i_0; s0 <= R.xy_i_1;)
	{
		const int m = s0 >> lm, mb = m << lm;
		const int s1 = min(R.xy_i_1, mb + (1 << lm) - 1);
		int nlo = 1 << 30, nhi = -1, zlo = 1 << 30, zhi = -1;
		for (int xyi = s0; xyi <= s1; xyi++)
		{
			DDSlice q;
			ddSlice<false>(im, R, pr, xyi, q);
			if (q.yx0 <= q.yx1 && q.zi0 <= q.zi1)
			{
				nlo = min(nlo, q.yx0);
				nhi = max(nhi, q.yx1);
				zlo = min(zlo, q.zi0);
				zhi = max(zhi, q.zi1);
			}
		}
		if (nhi >= 0)
		{
			for (int zt = zlo >> T.lz; zt <= zhi >> T.lz; zt++)
				for (int nt = nlo >> ln; nt <= nhi >> ln; nt++)
				{
					const int y0 = nt << ln, y1 = y0 + (1 << ln) - 1;
					const int z0 = zt << T.lz, z1 = z0 + (1 << T.lz) - 1;
					int first = -1, last = -1, vox = 0;
					for (int xyi = s0; xyi <= s1; xyi++)
					{
						DDSlice q;
						ddSlice<false>(im, R, pr, xyi, q);
						const int a0 = max(q.yx0, y0), a1 = min(q.yx1, y1);
						const int b0 = max(q.zi0, z0), b1 = min(q.zi1, z1);
						if (a0 <= a1 && b0 <= b1)
						{
							if (first < 0)
								first = xyi;
							last = xyi;
							vox += (a1 - a0 + 1) * (b1 - b0 + 1);
						}
					}
					if (vox > 0)
					{
						const int tx = R.flag_y ? nt : m, ty = R.flag_y ? m : nt;
						onRecord(((frame * T.ntz + zt) * T.nty + ty) * T.ntx + tx, 0.f,
						         (uint32_t)(first - mb) | ((uint32_t)(last - mb) << 6), vox);
					}
				}
		}
		s0 = s1 + 1;
	}
}

// (the loop's bound is uniform: a plan of few classes compares few cuts)
__device__ __forceinline__ int lengthClass(const DPlan& pl, int segs)
{
	int c = 0;
	for (int k = 0; k < pl.C - 1; k++)
		c += (segs >= pl.cut[k]) ? 1 : 0;
	return c;
}

// Each workgroup bins one contiguous range of rays (they are in locality
// order), so a bin's records from one workgroup come from neighbouring rays
// and the tile backprojection's reads of their ray-table entries coalesce.
// PASS 0: each workgroup counts the records of its rays per bin (LDS),
// keeps its counts in blockCnt[block][bin] and adds them to count[bin].
// PASS 1 (same grid, same rays per workgroup): each workgroup reserves its
// counts in every bin from cursor[bin] and walks its rays again, writing
// each record into its range (an LDS countdown per bin, so a record beyond
// the reservation is caught without a global read).  DD records have no
// alpha.
// LDS: cnt[nB] ints, then (PASS 1) base[nB] 32-bit record indices.
template <bool DD, bool TOF, bool S64, int PASS>
__global__ void __launch_bounds__(kBinThreads) kBin(DImage im, DProj pr, int64_t nRays, DTiles T,
                                            DPlan pl)
{
	extern __shared__ int sm[];
	const int nB = T.nTiles * pl.C;
	int* cnt = sm;
	uint32_t* base = reinterpret_cast<uint32_t*>(sm + nB);
	if (pl.listed != nullptr)
		nRays = min(nRays, max((int64_t)0, (int64_t)*pl.listed - pl.listFirst) * pl.R);
	const int64_t per = (nRays + gridDim.x - 1) / gridDim.x;
	const int64_t tEnd = min(nRays, (int64_t)(blockIdx.x + 1) * per);
	const int64_t t0 = (int64_t)blockIdx.x * per + threadIdx.x;
	const int64_t stride = blockDim.x;
	unsigned int* myCnt = pl.blockCnt + (int64_t)blockIdx.x * nB;
	auto binOne = [&](uint32_t t, auto&& onRecord) {
		if constexpr (DD)
			binRayDD(im, pr, T, pl.ray, t, onRecord);
		else
			binRay<TOF, S64>(im, pr.tof, T, pl.ray, t, pl.err, onRecord);
	};
	if (PASS == 0)
	{
		for (int i = threadIdx.x; i < nB; i += blockDim.x)
			cnt[i] = 0;
		__syncthreads();
		for (int64_t t = t0; t < tEnd; t += stride)
			binOne((uint32_t)t, [&](int tile, float, uint32_t, int segs) {
				atomicAdd(&cnt[tile * pl.C + lengthClass(pl, segs)], 1);
			});
		__syncthreads();
		for (int i = threadIdx.x; i < nB; i += blockDim.x)
		{
			myCnt[i] = (unsigned int)cnt[i];
			if (cnt[i] != 0)
				atomicAdd(&pl.count[i], (unsigned long long)cnt[i]);
		}
		return;
	}
	if (pl.skip != nullptr)
	{
		// read once for the workgroup: another one may be setting it now
		if (threadIdx.x == 0)
			cnt[0] = *pl.skip;
		__syncthreads();
		const int skip = cnt[0];
		__syncthreads();
		if (skip != 0)
			return;
	}
	for (int i = threadIdx.x; i < nB; i += blockDim.x)
	{
		const int c = (int)myCnt[i];
		base[i] = (c != 0) ? (uint32_t)(pl.tileOff[i] +
		                                (int64_t)atomicAdd(&pl.cursor[i], (unsigned int)c))
		                   : 0u;
		cnt[i] = c;
	}
	__syncthreads();
	for (int64_t t = t0; t < tEnd; t += stride)
		binOne((uint32_t)t, [&](int tile, float a0, uint32_t pv, int segs) {
			const int b = tile * pl.C + lengthClass(pl, segs);
			const int left = atomicSub(&cnt[b], 1);
			if (left > 0)
			{
				const int64_t j = (int64_t)base[b] + left - 1;
				// one record of consecutive words (one vector store)
				uint32_t* o = pl.rec + recWords(DD) * j;
				o[0] = (uint32_t)t;
				if (!DD)
					o[1] = __float_as_uint(a0);
				o[recWords(DD) - 1] = withFineClass(DD, pv, segs, T.tx + T.ty + T.tz);
			}
			else
				atomicOr(pl.err, 1);
		});
}

// Records of every chunk ordered by their fine length class (withFineClass),
// once when the plan is built: the tile backprojection's waves then take
// records of about the same length, where the plan's bins can hold only a
// few classes per tile.  Each window of kSortWin records of a chunk is
// sorted in place, stably by (class, position): one workgroup per chunk,
// each lane holding its records in registers between the reads and the
// writes; a record's rank in its class within a group of 64 is counted
// with wave ballots.  The tile sums do not depend on the records' order
// (fixed point), so the backprojection is unchanged.
constexpr int kSortWin = 2048;

template <bool DD>
__global__ void __launch_bounds__(256) kChunkSort(DPlan pl, const TileChunk* __restrict__ chunks)
{
	constexpr int G = kSortWin / 64, GPW = G / 4;  // groups of 64, per wave
	__shared__ int cntG[G][16];
	__shared__ int offG[G][16];
	__shared__ int base[16];
	const TileChunk ch = chunks[blockIdx.x];
	const int lane = (int)(threadIdx.x & 63u), wv = (int)(threadIdx.x >> 6);
	const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
	for (int w0 = 0; w0 < ch.count; w0 += kSortWin)
	{
		const int n = min(kSortWin, ch.count - w0);
		const int64_t j0 = ch.begin + w0;
		uint32_t k[GPW], v[GPW];
		uint32_t al[GPW];
		int cls[GPW];
#pragma unroll
		for (int i = 0; i < GPW; i++)
		{
			const int g = wv + 4 * i, r = g * 64 + lane;
			k[i] = 0u;
			v[i] = 0u;
			al[i] = 0u;
			cls[i] = 16;  // no record
			if (r < n)
			{
				const uint32_t* o = pl.rec + recWords(DD) * (j0 + r);
				k[i] = o[0];
				v[i] = o[recWords(DD) - 1];
				if (!DD)
					al[i] = o[1];
				cls[i] = fineClassOf(DD, v[i]);
			}
			for (int c = 0; c < 16; c++)
			{
				const int m = __popcll(__ballot(cls[i] == c));
				if (lane == 0)
					cntG[g][c] = m;
			}
		}
		__syncthreads();
		if (threadIdx.x < 16)
		{
			const int c = (int)threadIdx.x;
			int sum = 0;
			for (int g = 0; g < G; g++)
			{
				offG[g][c] = sum;
				sum += cntG[g][c];
			}
			base[c] = sum;
		}
		__syncthreads();
		if (threadIdx.x == 0)
		{
			int sum = 0;
			for (int c = 0; c < 16; c++)
			{
				const int t = base[c];
				base[c] = sum;
				sum += t;
			}
		}
		__syncthreads();
#pragma unroll
		for (int i = 0; i < GPW; i++)
		{
			const int g = wv + 4 * i;
			uint64_t mine = 0ull;
			for (int c = 0; c < 16; c++)
			{
				const uint64_t m = __ballot(cls[i] == c);
				if (cls[i] == c)
					mine = m;
			}
			if (cls[i] < 16)
			{
				const int64_t j = j0 + base[cls[i]] + offG[g][cls[i]] + __popcll(mine & below);
				uint32_t* o = pl.rec + recWords(DD) * j;
				o[0] = k[i];
				if (!DD)
					o[1] = al[i];
				o[recWords(DD) - 1] = v[i];
			}
		}
		__syncthreads();
	}
}

hipError_t launchChunkSort(bool dd, const DPlan& pl, const TileChunk* chunks, int64_t nChunks,
                           hipStream_t st)
{
	for (int64_t c0 = 0; c0 < nChunks; c0 += 65535)
	{
		const unsigned g = (unsigned)std::min<int64_t>(65535, nChunks - c0);
		if (dd)
			kChunkSort<true><<<g, 256, 0, st>>>(pl, chunks + c0);
		else
			kChunkSort<false><<<g, 256, 0, st>>>(pl, chunks + c0);
	}
	return hipGetLastError();
}

// One chunk: accumulate its ray pieces in the LDS tile `acc`, then add the
// tile into y (frame f of the chunk's tile).  v[e] is the value
// backprojected along LOR e (split over the rays as
// ProjectorSiddon::backProjection does, ProjectorSiddon.cpp:321-328); LORs
// with v == 0 are skipped.  Each lane runs a three-stage pipeline over its
// records: the fields of the record two ahead are read, the ray-table entry
// and value of the next one are in flight, and the current one is set up
// from its table entry and walked (the walk itself issues no global loads).
//
// Tile accumulation.  FP32 atomic adds into LDS run at about half a lane per
// clock per CU and bounded the kernel; 64-bit integer LDS atomics do not.
// So the tile is accumulated in fixed point, each contribution c = v/R * w
// rounded once to a multiple of 2^-k and added as an integer (exact and
// order-free, so the tile sum is deterministic); the flush converts back
// (int64 -> float, times 2^-k: exact scaling).  A voxel takes at most one
// contribution per record, so with every term below 2^lim in magnitude,
// lim = min(62 - e2, 51) (records < 2^e2; 2^51 for the conversion), no
// partial sum can overflow; a term that does not fit — and any non-finite
// one — is added to the image directly with a global FP32 atomic, as the
// direct backprojection does.  k is chosen from the launch's values: E, the
// binade of the median nonzero |v| (kVExpScale), 2^10 of headroom,
// and wmax, the largest segment weight (voxel diagonal, times the TOF norm):
// k = lim - (E + 10 + ew), wmax < 2^ew.
// Typical contributions then keep ~35 bits below their magnitude; values
// more than ~1000 times the median (the heavy tail of EM ratios m / Ax on
// LORs with tiny projections) cost a global atomic instead of precision.
// The scale only trades precision against that fallback: no choice of it
// can overflow the tile.  The 32^3 shape (whose 64-bit tile would need
// 256 KB of LDS) accumulates in FP32.
//
// SUM64: the tile is summed in FP64 instead (ds_add_f64: any term, no scale,
// sums good to 2^-53 of their largest partial sum, rounded once at the flush):
// DD, and calls without a plan (pl.vexp null), whose FP32 atomics kept 24 bits
// of every term: one 2^-15 of the fixed-point scale and smaller keeps fewer, one
// below 2^-39 none.  An EM subset of 2 M corrected LORs into 181 x 173 x 109
// takes 4.08 ms so (fixed point: 3.83; atomics: 35.4), 1 M TOF LORs x 4 rays
// forward and back at 200 x 200 x 128 2.22 (2.08; 20.5).
//
// DD records (DD = true) hold the LOR alone: its table entry (ddEntry) is set
// up (ddSetup) and its footprint swept over the slices, minor-axis voxels and
// z planes of the tile (ddVisit), the voxel weights exactly those of the
// direct sweep.  A footprint's weights have no bound of a few instructions, and
// the per-term range test and its global atomic, in fixed point, cost more
// than the slower FP64 LDS add (4 M bins of 16 frames at 128 x 128 x 96,
// projection PSF: 28.2 -> 14.1 ms, with the PSF segment table 34.5 before).
// Planned Siddon, with more adds an instruction, would lose by it: 6.0 -> 7.5
// ms for 10 M TOF LORs x 4 rays.
// The projector's PSF segment tables of one direction (flip: the
// backprojection's), made in the workgroup's dynamic LDS (DPsf::ldsBytes,
// given by the DD kernels' launches) by all its threads; the caller waits at
// a barrier before reading them.  Returns the LDS tables, or null when the
// projector's stay in global memory.
__device__ __forceinline__ const float4* psfStage(const DPsf& P, bool flip, float4* l)
{
	if (P.ldsBytes == 0)
		return nullptr;
	const int ns = psfSegments(P.K);
	const double* c = flip ? P.cumFlip : P.cum;
	const float* k = flip ? P.kflip : P.k;
	for (int i = threadIdx.x; i < P.numS * ns; i += blockDim.x)
	{
		const int row = i / ns;
		psfSegment(k + row * psfRowTaps(P.K), c + row * (P.K + 2), P.K, i - row * ns, l + i);
	}
	return l;
}

template <bool DD, bool TOF, bool S64, int SHAPE, bool SUM64>
__device__ __forceinline__ void tileChunk(const KArgs& a, const DTiles& T,
                                          const DPlanRead& pl, const TileChunk ch,
                                          const float* __restrict__ v,
                                          float* __restrict__ y, unsigned long long* acc64,
                                          const float4* psfL)
{
	float* acc = reinterpret_cast<float*>(acc64);
	constexpr int TX = tileDim(SHAPE, 0), TY = tileDim(SHAPE, 1), TZ = tileDim(SHAPE, 2);
	constexpr int NV = TX * TY * TZ, NT = tileThreads(SHAPE);
	int t = ch.tile;
	const int txi = t % T.ntx;
	t /= T.ntx;
	const int tyi = t % T.nty;
	t /= T.nty;
	const int tzi = t % T.ntz;
	const int f = t / T.ntz;
	WalkBox B;
	B.x0 = txi * TX;
	B.y0 = tyi * TY;
	B.z0 = tzi * TZ;
	B.x1 = min(B.x0 + TX, a.im.nx);
	B.y1 = min(B.y0 + TY, a.im.ny);
	B.z1 = min(B.z0 + TZ, a.im.nz);
	// voxel index in bytes of the LDS tile's words (8: fixed point, 4: FP32)
	auto wordBytes = [&](int esz) {
		B.sx = esz;
		B.sy = TX * esz;
		B.sz = TX * TY * esz;
		B.base = -(B.z0 * B.sz + B.y0 * B.sy + B.x0 * B.sx);
	};
	constexpr int NW = (SHAPE == 2) ? NV / 2 : NV;  // 64-bit words of the LDS tile
	for (int i = threadIdx.x; i < NW; i += NT)
		acc64[i] = 0ull;
	// fixed-point scale of this chunk (uniform)
	int fixed = 0, k = 0;
	float climit = 0.f, wbound = 0.f;
	if constexpr (SHAPE != 2 && !SUM64)
	{
		{
			// largest voxel weight: a segment is at most the voxel diagonal
			float wmax = 1.01f * sqrtf(a.im.vx * a.im.vx + a.im.vy * a.im.vy +
			                           a.im.vz * a.im.vz);
			if (TOF)
				wmax *= 1.01f * a.pr.tof.norm;
			int ew = 0;
			(void)frexpf(wmax, &ew);
			// terms below 2^lim, lim = min(62 - e2, 51): no partial sum of
			// the chunk's at most 2^e2 terms overflows, and every term
			// converts exactly through the 2^52 bias below
			const int e2 = 32 - __clz(ch.count);
			const int lim = min(62 - e2, 51);
			k = lim - (*pl.vexp + 10 + ew);
			// |c| < 2^(lim - k) <=> |c * 2^k| < 2^lim (inf when above the
			// float range: then every finite c qualifies)
			climit = ldexpf(1.f, lim - k);
			wbound = wmax;
			fixed = 1;
		}
	}
	fixed = __builtin_amdgcn_readfirstlane(fixed);
	k = __builtin_amdgcn_readfirstlane(k);
	float* yf = y + (int64_t)f * a.im.nvox;
	__syncthreads();
	const uint32_t R = (uint32_t)pl.R;
	const bool rPow2 = (R & (R - 1u)) == 0u;
	const int rShift = __ffs((int)R) - 1;
	const float rInvPow2 = ldexpf(1.f, -rShift);
	const uint64_t nRays = (uint64_t)a.L.n * R;
	// no record (keys are < n * R < 2^32); a key is checked against n * R
	// where it is used, not where it is read, so that its load stays in
	// flight during the walk
	constexpr uint32_t kNone = 0xffffffffu;
	auto lorOf = [&](uint32_t key) { return rPow2 ? key >> rShift : key / R; };
	struct Rec
	{
		uint32_t key, pv;
		float al;
	};
	// Siddon: the ray's end points and frame (two float4), with the FP32
	// set-up two more (sidStore); DD: kDDVec (ddStore)
	constexpr int NE = DD ? kDDVec : rayTabVec(S64);
	struct Ray
	{
		float4 e[NE];
		float val;
	};
	auto readRecord = [&](int k, Rec& r) {
		r.key = kNone;
		r.al = 0.f;
		r.pv = 0u;
		if (k < ch.count)
		{
			const int64_t j = ch.begin + k;
			const uint32_t* o = pl.rec + recWords(DD) * j;
			r.key = o[0];
			if (!DD)
				r.al = __uint_as_float(o[1]);
			r.pv = o[recWords(DD) - 1];
		}
	};
	auto readRay = [&](uint32_t key, Ray& q) {
#pragma unroll
		for (int i = 0; i < NE; i++)
			q.e[i] = make_float4(0.f, 0.f, 0.f, 0.f);
		q.val = 0.f;
		if ((uint64_t)key < nRays)
		{
#pragma unroll
			for (int i = 0; i < NE; i++)
				q.e[i] = pl.ray[NE * (uint64_t)key + i];
			q.val = v[DD ? key : lorOf(key)];
		}
	};
	// Siddon: a record whose value times the largest term factor (wmax:
	// every term c = v * w of its walk is at most |v| * wmax) is within
	// the fixed-point range walks with `addIn`, which skips the per-term
	// range test; other records (and the FP32 tile) walk with `add`
	auto walk = [&](const Rec& rc, const Ray& q, auto&& add, auto&& addIn, auto inRange) {
		float val = q.val;
		if ((uint64_t)rc.key >= nRays || val == 0.f)
			return;
		{
			const float4 qa = q.e[0], qb = q.e[1];
			if ((S64 ? __float_as_int(qb.w) : (int)(__float_as_uint(qb.w) & 0xffffu)) != f)
				return;
			const float3 q1 = make_float3(qa.x, qa.y, qa.z), q2 = make_float3(qa.w, qb.x, qb.y);
			// v / R: for R a power of two the product with 1/R is the same
			// correctly rounded value (1/R exact), one multiply
			if (R > 1u)
				val = rPow2 ? val * rInvPow2 : val / (float)R;
			const uint32_t pv = rc.pv;
			const int vx = B.x0 + (int)(pv & 31u), vy = B.y0 + (int)((pv >> 5) & 31u),
			          vz = B.z0 + (int)((pv >> 10) & 31u);
			const int dx = (int)((pv >> 15) & 15u) - 8, dy = (int)((pv >> 19) & 15u) - 8,
			          dz = (int)((pv >> 23) & 15u) - 8;
			// FP32 set-up: every record, a ray's first included (its voxel is
			// the walk's first, its alpha the ray's start), is re-entered from
			// the ray's stored set-up, one instruction stream for the wave;
			// FP64 set-up: the first record walks from the ray's entry
			const bool entry = S64 && (pv >> 31) != 0;
			if (!entry && (vx >= B.x1 || vy >= B.y1 || vz >= B.z1))
				return;
			SidRay s;
			if (!S64)
				sidLoad(q1, q2, q.e[2 % NE], q.e[3 % NE], s);
			else if (!sidSetup<TOF, S64>(a.im, q1, q2, a.pr.tof, qb.z, s))
				return;
			if (!entry)
				sidRestart<S64>(a.im, s, rc.al, vx, vy, vz, dx, dy, dz);
			const float vs = val * s.ws;
			auto go = [&](auto&& fn) {
				sidWalk<TOF, S64>(a.im, s, a.pr.tof, B, entry, vx, vy, vz,
				                  [&](int gx, int gy, int gz, uint32_t idx, float, float w,
				                      uint32_t) { fn(idx, gx, gy, gz, vs * w); });
			};
			if constexpr (decltype(inRange)::value)
			{
				if (fabsf(val) * wbound < climit)
					go(addIn);
				else
					go(add);
			}
			else
				go(add);
		}
	};
	// DD: a wave's 64 records are swept one (record, slice) pair per lane.
	// The pairs are numbered by the wave's prefix sum of the records' slice
	// counts (last - first + 1 of the record's word), and the lane of pair s
	// finds its record, the last whose first pair is at most s, by a binary
	// search over the prefix sums; so the lanes differ in the footprint of
	// their slice only, not in their record's number of slices.  Each pair
	// reads its LOR's set-up (the pairs of one record read the same lines in
	// one load).  The sums and searches run in the wave's uniform control
	// flow (the trip counts are wave-uniform), with no workgroup barrier.
	auto pipelineDD = [&](auto&& add) {
		const int lane = (int)(threadIdx.x & 63u);
		for (int i0 = (int)threadIdx.x - lane; i0 < ch.count; i0 += NT)
		{
			Rec rc;
			readRecord(i0 + lane, rc);
			const int ns = (uint64_t)rc.key < nRays
			                   ? (int)((rc.pv >> 6) & 63u) - (int)(rc.pv & 63u) + 1
			                   : 0;
			int incl = ns;
#pragma unroll
			for (int d = 1; d < 64; d <<= 1)
			{
				const int t = __shfl_up(incl, (unsigned int)d, 64);
				if (lane >= d)
					incl += t;
			}
			const int excl = incl - ns;
			const int total = __shfl(incl, 63, 64);
			for (int s0 = 0; s0 < total; s0 += 64)
			{
				const int s = s0 + lane;
				int r = 0;
#pragma unroll
				for (int b = 32; b > 0; b >>= 1)
					r += (__shfl(excl, r + b, 64) <= s) ? b : 0;
				const uint32_t key = (uint32_t)__shfl((int)rc.key, r, 64);
				const uint32_t pv = (uint32_t)__shfl((int)rc.pv, r, 64);
				const int slot = s - __shfl(excl, r, 64);
				if (s >= total)
					continue;
				const float val = v[key];
				float4 e[kDDVec];
#pragma unroll
				for (int j = 0; j < kDDVec; j++)
					e[j] = pl.ray[kDDVec * (uint64_t)key + j];
				if (val == 0.f || ddFrame(e[5]) != f)
					continue;
				DDRay D;
				ddLoad(a.im, a.pr, e, true, D);
				// the pair's slice: first + slot of the tile's slab
				const int xyi = (D.flag_y ? B.y0 : B.x0) + (int)(pv & 63u) + slot;
				if (xyi >= (D.flag_y ? B.y1 : B.x1))
					continue;
				const int ylo = D.flag_y ? B.x0 : B.y0, yhi = (D.flag_y ? B.x1 : B.y1) - 1;
				auto sweep = [&](const DDRay& Q, auto tab) {
					ddVisit<TOF, decltype(tab)::value>(
					             a.im, Q, a.pr, xyi, xyi, ylo, yhi, B.z0, B.z1 - 1,
					             [&](int, int xs, int yxi, int zi, float w) {
						             const int gx = Q.flag_y ? yxi : xs,
						                       gy = Q.flag_y ? xs : yxi;
						             add((uint32_t)(B.base + zi * B.sz + gy * B.sy + gx * B.sx),
						                 gx, gy, zi, val * w);
					             });
				};
				// (two copies of the sweep: one reads the PSF segments from LDS)
				if (psfL != nullptr)
				{
					D.ptab = psfL + D.psfRow * psfSegments(a.pr.psf.K);
					sweep(D, std::true_type{});
				}
				else
					sweep(D, std::false_type{});
			}
		}
	};
	auto pipeline = [&](auto&& add, auto&& addIn, auto inRange) {
		if constexpr (DD)
			pipelineDD(add);
		else
		{
			int i = threadIdx.x;
			Rec r0, r1;
			Ray q0;
			readRecord(i, r0);
			readRay(r0.key, q0);
			readRecord(i + NT, r1);
			for (; i < ch.count; i += NT)
			{
				Ray q1;
				readRay(r1.key, q1);
				Rec r2;
				readRecord(i + 2 * NT, r2);
				walk(r0, q0, add, addIn, inRange);
				r0 = r1;
				q0 = q1;
				r1 = r2;
			}
		}
	};
	// c * 2^k rounded to an integer: one FP64 fma with the bias 1.5 * 2^52
	// (|c * 2^k| < 2^51, so the sum stays in [2^52, 2^53), whose ulp is 1:
	// the fma's rounding is the round-to-nearest-even of c * 2^k, which is
	// exact in FP64), the integer being the sum's bits less the bias's.
	// The bias's low word is zero, so that is one 32-bit subtract.
	const double scale = ldexp(1.0, k);
	constexpr double kBias = 6755399441055744.0;  // 1.5 * 2^52
	constexpr unsigned long long kBiasBits = 0x4338000000000000ull;
	if constexpr (SUM64)
	{
		wordBytes(8);
		auto addD = [&](uint32_t idx, int, int, int, float c) {
			__hip_atomic_fetch_add(
			    reinterpret_cast<double*>(reinterpret_cast<char*>(acc64) + idx), (double)c,
			    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
		};
		pipeline(addD, addD, std::integral_constant<bool, false>{});
	}
	else if (fixed)
	{
		wordBytes(8);
		auto addFixed = [&](uint32_t idx, float c) {
			const double d = fma((double)c, scale, kBias);
			ldsAdd64(reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(acc64) + idx),
			         (long long)((unsigned long long)__double_as_longlong(d) - kBiasBits));
		};
		pipeline(
		    [&](uint32_t idx, int gx, int gy, int gz, float c) {
			    if (fabsf(c) < climit)
				    addFixed(idx, c);
			    else  // out of the fixed-point range, or not finite
				    unsafeAtomicAdd(yf + (int64_t)gz * a.im.nxy + (int64_t)gy * a.im.nx + gx, c);
		    },
		    [&](uint32_t idx, int, int, int, float c) { addFixed(idx, c); },
		    std::true_type{});
	}
	else
	{
		wordBytes(4);
		auto addFloat = [&](uint32_t idx, int, int, int, float c) {
			ldsAdd(reinterpret_cast<float*>(reinterpret_cast<char*>(acc) + idx), c);
		};
		pipeline(addFloat, addFloat, std::integral_constant<bool, false>{});
	}
	__syncthreads();
	for (int i = threadIdx.x; i < NV; i += NT)
	{
		const int lx = i % TX, ly = (i / TX) % TY, lz = i / (TX * TY);
		const int gx = B.x0 + lx, gy = B.y0 + ly, gz = B.z0 + lz;
		float s;
		if constexpr (SUM64)
			s = (float)__longlong_as_double((long long)acc64[i]);
		else
			s = fixed ? ldexpf((float)(long long)acc64[i], -k) : acc[i];
		if (s != 0.f && gx < B.x1 && gy < B.y1 && gz < B.z1)
			unsafeAtomicAdd(yf + (int64_t)gz * a.im.nxy + (int64_t)gy * a.im.nx + gx, s);
	}
	__syncthreads();  // acc is reused by the next chunk
}

// Waves a SIMD that a DD tile's LDS leaves room for (16^3 and 32 x 32 x 8: 16 a
// CU and more); at 131 registers one 32 x 32 x 8 workgroup a CU was left of two
// (150 k TOF LORs with a PSF at 95 x 97 x 47, forward and back: 1.29 ms, now 1.14).
__host__ __device__ constexpr int kDDTileWaves(int shape)
{
	return shape == 1 ? 2 : 4;
}

// One workgroup per chunk (pl.queue == null), or a persistent grid taking
// chunks from the plan's queue until it is empty.  Every workgroup leaves
// once the queue index passes the chunk count, so the grid always drains.
template <bool DD, bool TOF, bool S64, int SHAPE, bool SUM64>
__global__ void __launch_bounds__(tileThreads(SHAPE))
    __attribute__((amdgpu_waves_per_eu(DD ? kDDTileWaves(SHAPE) : tileThreads(SHAPE) / 256, 8)))
    kTileBack(KArgs a, DTiles T, DPlanRead pl, const float* __restrict__ v,
              float* __restrict__ y)
{
	// NV 64-bit words (fixed point or FP64), or NV floats for the 32^3 shape
	constexpr int NV = tileDim(SHAPE, 0) * tileDim(SHAPE, 1) * tileDim(SHAPE, 2);
	__shared__ unsigned long long acc[SHAPE == 2 ? NV / 2 : NV];
	extern __shared__ float4 psfLds[];
	const float4* psfL = nullptr;
	if constexpr (DD)
	{
		psfL = psfStage(a.pr.psf, true, psfLds);
		__syncthreads();
	}
	if (pl.queue == nullptr)
	{
		tileChunk<DD, TOF, S64, SHAPE, SUM64>(a, T, pl, pl.chunks[blockIdx.x], v, y, acc, psfL);
		return;
	}
	if (pl.err != nullptr && *pl.err != 0)
		return;
	const int64_t nChunks = pl.nChunksDev != nullptr ? *pl.nChunksDev : pl.nChunks;
	// the next chunk's index is passed through the tile's first word (read
	// between two barriers, before the chunk clears the tile), so the
	// workgroup's LDS is the tile alone: 32 KB for 16^3, five per CU
	for (;;)
	{
		if (threadIdx.x == 0)
			acc[0] = (unsigned long long)atomicAdd(&pl.queue[0], 1u);
		__syncthreads();
		const int64_t c = (int64_t)acc[0];
		__syncthreads();
		if (c >= nChunks)
			break;
		tileChunk<DD, TOF, S64, SHAPE, SUM64>(a, T, pl, pl.chunks[c], v, y, acc, psfL);
	}
	if (threadIdx.x == 0)
	{
		__threadfence();
		if (atomicAdd(&pl.queue[1], 1u) == gridDim.x - 1)
		{
			atomicExch(&pl.queue[0], 0u);
			atomicExch(&pl.queue[1], 0u);
		}
	}
}

// EM ratio per LOR (computeEMUpdateImage, OSEM_CPU.cpp:329-374): the
// forward projection of x, corrected, against the measurement; v[e] = 0
// where the LOR is skipped (zero measurement / factor, invalid LOR, or a
// denominator at or below the threshold).
// The hardware deals workgroups to the XCDs round-robin (workgroup b runs on
// XCD b % kXcds).  With the grid a multiple of kXcds, workgroup b takes the
// range (b % kXcds) * (grid / kXcds) + b / kXcds instead, so each XCD works
// through one contiguous stretch of the LORs: in locality order their voxels
// then share that XCD's L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int64_t xcdRange(int64_t b, int64_t grid)
{
	return (b % kXcds) * (grid / kXcds) + b / kXcds;
}

// The EM ratio of LOR e from its forward projection s (summed over its rays).
__device__ __forceinline__ float emRatioOut(const KArgs& a, int64_t e, float s, float m,
                                           float sf, float af)
{
	float upd = (a.pr.numRays > 1) ? s / (float)a.pr.numRays : s;
	if (a.plain)
		return upd;
	if (a.c.sens)
		upd *= sf;
	if (a.c.att)
		upd *= af;
	upd *= a.c.g;
	if (a.c.randoms)
		upd += a.c.randoms[e];
	if (a.c.scatter)
		upd += a.c.scatter[e];
	// in-vivo attenuation precorrection (OSEM_GPU.cu:1303-1308)
	if (a.c.precorr)
		upd *= a.c.precorr[e];
	float out = 0.f;
	if (fabsf(upd) > a.c.denomThr)
	{
		out = m / upd;
		if (a.c.sens)
			out *= sf;
		if (a.c.att)
			out *= af;
		out *= a.c.g;
	}
	return out;
}

// The line integral of an FP32 ray's stretch `part` of PARTS (sidPart), by one
// of PARTS neighbouring lanes, all of them here with the same ray; it ends where
// the next one starts.
template <bool TOF, bool BRICK, int PARTS>
__device__ __forceinline__ float siddonPart(const DImage& P, const float* __restrict__ img,
                                            float3 p1, float3 p2, const DTof& tof, float tofv,
                                            int part)
{
	SidRay r;
	int vx, vy, vz, dx, dy, dz;
	auto outside = [&]() {
		return (unsigned)vx >= (unsigned)P.nx || (unsigned)vy >= (unsigned)P.ny ||
		       (unsigned)vz >= (unsigned)P.nz;
	};
	if (!sidSetup<TOF, false>(P, p1, p2, tof, tofv, r) ||
	    !sidFirst<false>(P, r, vx, vy, vz, dx, dy, dz) || outside())
		return 0.f;
	const float start = part > 0 ? sidPart(P, r, part, PARTS, vx, vy, vz, dx, dy, dz) : r.a_cur;
	const float next = __shfl_down(start, 1, PARTS);
	if (part < PARTS - 1)
		r.amax = next;
	if (!(start < r.amax) || outside())
		return 0.f;
	sidRestart<false>(P, r, start, vx, vy, vz, dx, dy, dz);
	return sidForward<TOF, false, BRICK>(P, r, tof, img, false, vx, vy, vz) * r.ws;
}

// Siddon: LPE lanes per LOR splitting its rays, made from the resolved LOR
// (the LUT stays in L2; a plan's ray table, read from HBM, measured slower).
// BRICK: gathers from the bricked copy of x (a.xb; useBricks), else from x.
// PARTS: lanes per ray, in turn along it (kSplitRays; the FP32 set-up's).
// LIST: of listed LORs (KArgs::list; two registers more, which at 96 spill).
template <bool TOF, int LPE, bool S64, bool BRICK, int PARTS, bool LIST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(S64 ? 4 : 5, 8)))
kEmRatio(KArgs a, float* __restrict__ v)
{
	constexpr int lanes = LPE * PARTS;
	const int64_t total = (LIST ? lorCount(a) : a.L.n) * lanes;
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t t = xcdRange(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; t < total;
	     t += stride)
	{
		const int64_t e = LIST ? lorElement(a, t / lanes) : t / lanes;
		const int lane = (int)(t & (lanes - 1));
		const Lor l = fetchLor(a.sc, a.L, e, a.im.nt);
		const float m = a.c.meas ? a.c.meas[e] : 1.0f;
		const float sf = a.c.sens ? a.c.sens[e] : 1.0f;
		const float af = a.c.att ? a.c.att[e] : 1.0f;
		const bool skip = (m == 0.f || sf == 0.f || af == 0.f || l.frame < 0);
		float s = 0.f;
		if (!skip)
		{
			const float* img = BRICK ? a.xb + (int64_t)l.frame * a.bvox
			                         : a.x + (int64_t)l.frame * a.im.nvox;
			for (int r = lane / PARTS; r < a.pr.numRays; r += LPE)
			{
				float3 q1, q2;
				rayLine(a.pr, l, r, q1, q2);
				q1 = make_float3(q1.x - a.im.ox, q1.y - a.im.oy, q1.z - a.im.oz);
				q2 = make_float3(q2.x - a.im.ox, q2.y - a.im.oy, q2.z - a.im.oz);
				uint32_t c = 0;
				if constexpr (PARTS > 1)
					s += siddonPart<TOF, BRICK, PARTS>(a.im, img, q1, q2, a.pr.tof, l.tof,
					                                   lane & (PARTS - 1));
				else
					s += siddonRay<MODE_FWD, TOF, S64, BRICK>(a.im, const_cast<float*>(img), q1,
					                                          q2, 0.f, a.pr.tof, l.tof, c);
			}
		}
#pragma unroll
		for (int o = 1; o < lanes; o <<= 1)
			s += __shfl_xor(s, o, lanes);
		if (lane == 0)
			v[LIST ? t / lanes : e] = skip ? 0.f : emRatioOut(a, e, s, m, sf, af);
	}
}

// DD: LPE lanes per LOR, its set-up read from the plan's table (TAB) or made
// from the resolved LOR.  BRICK: gathers from the bricked copy of x, as the
// Siddon forward: a brick serves 4 slices of the sweep whichever the major
// axis, where rows along x serve one of y (4 M bins of 16 frames at 128 x 128 x 96:
// 15.8 -> 12.1 ms).
// LPE: lanes per LOR, each on every LPE-th slice (a lane per LOR leaves the
// chip idle in calls of few LORs: the forward of 150 k TOF LORs of 95 x 97 x
// 47 with a PSF 0.49 -> 0.40 ms); one where there are LORs enough.
// Four waves a SIMD where that needs no spill.
// LIST: as for Siddon.
template <bool TOF, bool S64, bool TAB, bool BRICK, int LPE, bool LIST>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu((TAB || (!S64 && BRICK)) ? 4 : 1, 8)))
kEmRatioDD(KArgs a, float* __restrict__ v)
{
	extern __shared__ float4 psfLds[];
	const float4* psfL = psfStage(a.pr.psf, false, psfLds);
	__syncthreads();
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	const int64_t total = (LIST ? lorCount(a) : a.L.n) * LPE;
	for (int64_t t = xcdRange(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; t < total;
	     t += stride)
	{
		const int64_t i = t / LPE, e = LIST ? lorElement(a, i) : i;
		const int lane = (int)(t & (LPE - 1));
		const float m = a.c.meas ? a.c.meas[e] : 1.0f;
		const float sf = a.c.sens ? a.c.sens[e] : 1.0f;
		const float af = a.c.att ? a.c.att[e] : 1.0f;
		int frame;
		Lor l;
		float4 de[kDDVec];
		if (TAB)
		{
			de[5] = a.rays[kDDVec * i + 5];
			frame = ddFrame(de[5]);
		}
		else
		{
			l = fetchLor(a.sc, a.L, e, a.im.nt);
			frame = l.frame;
		}
		const bool skip = (m == 0.f || sf == 0.f || af == 0.f || frame < 0);
		float s = 0.f;
		if (!skip)
		{
			DDRay D;
			if (TAB)
			{
#pragma unroll
				for (int k = 0; k < kDDVec; k++)
					if (k != 5)
						de[k] = a.rays[kDDVec * i + k];
				ddLoad(a.im, a.pr, de, false, D);
			}
			else
			{
				const float3 d1 = make_float3(l.p1.x - a.im.ox, l.p1.y - a.im.oy, l.p1.z - a.im.oz);
				const float3 d2 = make_float3(l.p2.x - a.im.ox, l.p2.y - a.im.oy, l.p2.z - a.im.oz);
				ddSetup<TOF, S64>(a.im, d1, d2, l.n1, l.n2, a.pr, l.tof, false, D);
			}
			const float* img = BRICK ? a.xb + (int64_t)frame * a.bvox
			                         : a.x + (int64_t)frame * a.im.nvox;
			// (two copies of the sweep: one reads the PSF segments from LDS)
			if (psfL != nullptr)
			{
				D.ptab = psfL + D.psfRow * psfSegments(a.pr.psf.K);
				s = ddSweepFwd<TOF, true, BRICK>(a.im, img, D, a.pr, lane, LPE);
			}
			else
				s = ddSweepFwd<TOF, false, BRICK>(a.im, img, D, a.pr, lane, LPE);
		}
#pragma unroll
		for (int o = 1; o < LPE; o <<= 1)
			s += __shfl_xor(s, o, LPE);
		if (lane == 0)
			v[i] = skip ? 0.f : emRatioOut(a, e, s, m, sf, af);
	}
}

// Sensitivity value per LOR (generateSensImage, OSEM_CPU.cpp:146-156):
// v[e] = sens factor * exp(-0.1 * Siddon(mu)) (Corrector.cpp:601-611).
// BRICK: mu from the attenuation image's bricked copy (a.xb), each XCD on one
// stretch of the LORs, as the EM ratio.  8.4 M LORs at 256 x 256 x 128: 4.1
// -> 3.1 ms, waiting on the gathers.
template <bool S64, bool BRICK>
__global__ void __launch_bounds__(256) kSensValue(KArgs a, float* __restrict__ v)
{
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t e = xcdRange(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; e < a.L.n;
	     e += stride)
	{
		const Lor l = fetchLor(a.sc, a.L, e, 1);
		float val = a.vals ? a.vals[e] : 1.0f;
		if (a.att)
		{
			uint32_t c2 = 0;
			const float mu = siddonRay<MODE_FWD, false, S64, BRICK>(
			    a.attIm, const_cast<float*>(BRICK ? a.xb : a.att), l.p1, l.p2, 0.f, a.pr.tof, 0.f,
			    c2);
			val *= expf(-mu * 0.1f);
		}
		v[e] = (l.frame >= 0) ? val : 0.f;
	}
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <bool DD, bool TOF, bool S64>
static hipError_t binT(int pass, const KArgs& a, const DTiles& T,
                       const DPlan& pl, int grid, hipStream_t st)
{
	const int nB = T.nTiles * pl.C;
	const int64_t nRays = a.L.n * (int64_t)pl.R;
	if (pass == 0)
		kBin<DD, TOF, S64, 0><<<grid, kBinThreads, (size_t)nB * sizeof(int), st>>>(a.im, a.pr, nRays,
		                                                                    T, pl);
	else
		kBin<DD, TOF, S64, 1><<<grid, kBinThreads, binLdsBytes(nB), st>>>(a.im, a.pr, nRays, T, pl);
	return hipGetLastError();
}

hipError_t launchRayPrep(const KArgs& a, float4* tab, int* err, hipStream_t st)
{
	const int64_t total = a.L.n * (int64_t)a.pr.numRays;
	if (total == 0)
		return hipSuccess;
	const unsigned g = (unsigned)std::min<int64_t>(std::max<int64_t>((total + 255) / 256, 1), 65536);
	// Siddon: the FP64 set-up stores the end points only (two float4 per
	// ray); the FP32 set-up stores its set-up too (four), with the TOF
	// constants when the projector has TOF
	if (a.pr.type != 1)
	{
		if (a.pr.setup64)
			kRayPrep<false, false, true><<<g, 256, 0, st>>>(a, tab, err);
		else if (a.pr.useTof)
			kRayPrep<false, true, false><<<g, 256, 0, st>>>(a, tab, err);
		else
			kRayPrep<false, false, false><<<g, 256, 0, st>>>(a, tab, err);
	}
	else if (a.pr.useTof)
	{
		if (a.pr.setup64)
			kRayPrep<true, true, true><<<g, 256, 0, st>>>(a, tab, err);
		else
			kRayPrep<true, true, false><<<g, 256, 0, st>>>(a, tab, err);
	}
	else
	{
		if (a.pr.setup64)
			kRayPrep<true, false, true><<<g, 256, 0, st>>>(a, tab, err);
		else
			kRayPrep<true, false, false><<<g, 256, 0, st>>>(a, tab, err);
	}
	return hipGetLastError();
}

template <bool DD>
static hipError_t binKind(int pass, const KArgs& a, const DTiles& T, const DPlan& pl,
                          int grid, hipStream_t st)
{
	const bool tof = a.pr.useTof != 0;
	if (a.pr.setup64)
		return tof ? binT<DD, true, true>(pass, a, T, pl, grid, st)
		           : binT<DD, false, true>(pass, a, T, pl, grid, st);
	return tof ? binT<DD, true, false>(pass, a, T, pl, grid, st)
	           : binT<DD, false, false>(pass, a, T, pl, grid, st);
}

hipError_t launchBin(int pass, const KArgs& a, const DTiles& T, const DPlan& pl,
                     int grid, hipStream_t st)
{
	return a.pr.type == 1 ? binKind<true>(pass, a, T, pl, grid, st)
	                      : binKind<false>(pass, a, T, pl, grid, st);
}

template <bool DD, bool TOF, bool S64, int SHAPE>
static void tileBackT(const KArgs& a, const DTiles& T, const DPlanRead& pl,
                      const float* v, float* y, unsigned grid, hipStream_t st)
{
	auto go = [&](auto k) {
		k<<<grid, tileThreads(SHAPE), DD ? a.pr.psf.ldsBytes : 0, st>>>(a, T, pl, v, y);
	};
	if constexpr (SHAPE == 2)
		go(kTileBack<DD, TOF, S64, SHAPE, false>);
	else if constexpr (DD)
		go(kTileBack<DD, TOF, S64, SHAPE, true>);
	else
		pl.vexp == nullptr ? go(kTileBack<DD, TOF, S64, SHAPE, true>)
		                   : go(kTileBack<DD, TOF, S64, SHAPE, false>);
}

template <bool DD, bool TOF, bool S64>
static void tileBackShape(const KArgs& a, const DTiles& T, const DPlanRead& pl,
                          const float* v, float* y, unsigned grid, hipStream_t st)
{
	switch (T.shape)
	{
	case 1:
		tileBackT<DD, TOF, S64, 1>(a, T, pl, v, y, grid, st);
		break;
	case 2:
		tileBackT<DD, TOF, S64, 2>(a, T, pl, v, y, grid, st);
		break;
	case 3:
		tileBackT<DD, TOF, S64, 3>(a, T, pl, v, y, grid, st);
		break;
	default:
		tileBackT<DD, TOF, S64, 0>(a, T, pl, v, y, grid, st);
		break;
	}
}

template <bool DD>
static void tileBackKind(const KArgs& a, const DTiles& T, const DPlanRead& pl,
                         const float* v, float* y, unsigned grid, hipStream_t st)
{
	const bool tof = a.pr.useTof != 0;
	if (a.pr.setup64)
	{
		if (tof)
			tileBackShape<DD, true, true>(a, T, pl, v, y, grid, st);
		else
			tileBackShape<DD, false, true>(a, T, pl, v, y, grid, st);
	}
	else
	{
		if (tof)
			tileBackShape<DD, true, false>(a, T, pl, v, y, grid, st);
		else
			tileBackShape<DD, false, false>(a, T, pl, v, y, grid, st);
	}
}

// *e = E, the binade of the median of the nonzero finite |v|: the smallest
// exponent with |v| < 2^E for at least half of them (|v| < 2^(b - 126) for
// biased exponent b); -126 when every value is zero or subnormal.
// Each workgroup counts the biased exponents of its values in LDS (8 copies:
// most values share a few exponents) and adds them to hist; the workgroup
// that finishes last picks E and clears hist and *done for the next launch.
// One launch, where clearing, counting and a serial scan of the 256 bins
// took three (22 us for 3000 values, of which the scan 17; now 4).
__global__ void __launch_bounds__(256) kVExpScale(const float* __restrict__ v, int64_t n,
                                                  unsigned int* hist, unsigned int* done, int* e)
{
	__shared__ unsigned int h[8][257];
	__shared__ unsigned long long s[257];
	__shared__ int last;
	const int t = (int)threadIdx.x;
#pragma unroll
	for (int k = 0; k < 8; k++)
		h[k][t] = 0u;
	__syncthreads();
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	int64_t i = (int64_t)blockIdx.x * blockDim.x + t;
	for (; i + 3 * stride < n; i += 4 * stride)
	{
		const float a0 = v[i], a1 = v[i + stride], a2 = v[i + 2 * stride], a3 = v[i + 3 * stride];
		atomicAdd(&h[t & 7][(__float_as_uint(a0) >> 23) & 0xffu], 1u);
		atomicAdd(&h[t & 7][(__float_as_uint(a1) >> 23) & 0xffu], 1u);
		atomicAdd(&h[t & 7][(__float_as_uint(a2) >> 23) & 0xffu], 1u);
		atomicAdd(&h[t & 7][(__float_as_uint(a3) >> 23) & 0xffu], 1u);
	}
	for (; i < n; i += stride)
		atomicAdd(&h[t & 7][(__float_as_uint(v[i]) >> 23) & 0xffu], 1u);
	__syncthreads();
	unsigned int c = 0u;
#pragma unroll
	for (int k = 0; k < 8; k++)
		c += h[k][t];
	if (c != 0u)
		atomicAdd(&hist[t], c);
	// the counts are in memory before this workgroup is counted as done (they
	// are read back by atomics too, so no fence, which would write the L2
	// back in every workgroup: 130 us for 10 M values)
	asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
	__syncthreads();
	if (t == 0)
		last = atomicAdd(done, 1u) == gridDim.x - 1;
	__syncthreads();
	if (!last)
		return;
	// s[t] = number of values of exponent t or above (1 .. 254)
	const unsigned int own = atomicExch(&hist[t], 0u);
	s[t] = (t >= 1 && t <= 254) ? own : 0u;
	if (t == 0)
	{
		s[256] = 0u;
		atomicExch(done, 0u);
	}
	__syncthreads();
#pragma unroll
	for (int d = 1; d < 256; d <<= 1)
	{
		const unsigned long long o = (t + d < 256) ? s[t + d] : 0u;
		__syncthreads();
		s[t] += o;
		__syncthreads();
	}
	const unsigned long long total = s[1];
	if (total == 0u)
	{
		if (t == 0)
			*e = -126;
	}
	else if (t >= 1 && 2u * s[t] >= total && 2u * s[t + 1] < total)
		*e = t - 126;
}

__global__ void __launch_bounds__(256) kClearWords(unsigned int* __restrict__ p, int64_t n)
{
	const int64_t stride = (int64_t)gridDim.x * blockDim.x;
	for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
		p[i] = 0u;
}

hipError_t launchClearWords(unsigned int* p, int64_t words, hipStream_t st)
{
	const unsigned g = (unsigned)std::min<int64_t>(std::max<int64_t>((words + 255) / 256, 1), 256);
	kClearWords<<<g, 256, 0, st>>>(p, words);
	return hipGetLastError();
}

// The LORs that an EM subset does not skip (m, sf and af, where given, not 0):
// one wave per stretch of the LORs (kListWaves of them), in order.
// PASS 0 counts each stretch's into part, kListScan makes them starts, PASS 1
// writes the list.
__device__ __forceinline__ int64_t listStretch(int64_t n)
{
	return ((n + kListWaves - 1) / kListWaves + 63) / 64 * 64;
}

template <int PASS>
__global__ void __launch_bounds__(256) kLorList(DCorr c, int64_t n, uint32_t* __restrict__ part,
                                                uint32_t* __restrict__ list)
{
	const int lane = (int)(threadIdx.x & 63u);
	const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), per = listStretch(n);
	const int64_t b = w * per, e = min(n, b + per);
	const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
	uint32_t at = PASS == 0 ? 0u : part[w];
	for (int64_t i0 = b; i0 < e; i0 += 256)
	{
		bool on[4];
#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			const int64_t i = min(i0 + 64 * k + lane, n - 1);
			on[k] = i0 + 64 * k + lane < e && !(c.meas && c.meas[i] == 0.f) &&
			        !(c.sens && c.sens[i] == 0.f) && !(c.att && c.att[i] == 0.f);
		}
#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			const uint64_t m = __ballot(on[k]);
			if (PASS == 1 && on[k])
				list[at + (uint32_t)__popcll(m & below)] = (uint32_t)(i0 + 64 * k + lane);
			at += (uint32_t)__popcll(m);
		}
	}
	if (PASS == 0 && lane == 0)
		part[w] = at;
}

// Exclusive prefix of v over the workgroup's 1024 threads; *total, its sum.
__device__ __forceinline__ unsigned long long scan1024(unsigned long long v,
                                                       unsigned long long* lds,
                                                       unsigned long long* total)
{
	const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
	unsigned long long incl = v;
#pragma unroll
	for (int d = 1; d < 64; d <<= 1)
	{
		const unsigned long long t = __shfl_up(incl, (unsigned int)d, 64);
		if (lane >= d)
			incl += t;
	}
	__syncthreads();
	if (lane == 63)
		lds[w] = incl;
	__syncthreads();
	unsigned long long before = 0, sum = 0;
#pragma unroll
	for (int k = 0; k < 16; k++)
	{
		before += (k < w) ? lds[k] : 0ull;
		sum += lds[k];
	}
	*total = sum;
	return before + incl - v;
}

__global__ void __launch_bounds__(1024)
    kStreamScan(DPlan pl, int64_t* __restrict__ tileOff, int nTiles, int64_t cap,
                TileChunk* __restrict__ chunks, StreamState* s)
{
	__shared__ unsigned long long lds[16];
	const int per = (nTiles + 1023) / 1024;
	const int t0 = min((int)threadIdx.x * per, nTiles), t1 = min(t0 + per, nTiles);
	auto tileCount = [&](int t) {
		unsigned long long n = 0;
		for (int k = 0; k < pl.C; k++)
			n += pl.count[t * pl.C + k];
		return n;
	};
	unsigned long long recs = 0;
	for (int t = t0; t < t1; t++)
		recs += tileCount(t);
	unsigned long long total, nFull, nPart;
	unsigned long long at = scan1024(recs, lds, &total);
	if (total > (unsigned long long)cap || s->err != 0)
	{
		if (threadIdx.x == 0)
		{
			s->nChunks = 0;
			if (total > (unsigned long long)cap)
				s->err |= 4;
		}
		return;
	}
	const unsigned long long CH = (unsigned long long)chunkRecords((int64_t)total);
	unsigned long long full = 0, part = 0;
	for (int t = t0; t < t1; t++)
	{
		const unsigned long long n = tileCount(t);
		full += n / CH;
		part += (n % CH != 0) ? 1 : 0;
	}
	unsigned long long fi = scan1024(full, lds, &nFull);
	unsigned long long pi = scan1024(part, lds, &nPart) + nFull;
	for (int t = t0; t < t1; t++)
	{
		const unsigned long long begin = at;
		for (int k = 0; k < pl.C; k++)
		{
			tileOff[t * pl.C + k] = (int64_t)at;
			at += pl.count[t * pl.C + k];
		}
		for (unsigned long long b = begin; b < at; b += CH)
		{
			TileChunk c;
			c.begin = (int64_t)b;
			c.tile = t;
			c.count = (int32_t)(at - b < CH ? at - b : CH);
			chunks[c.count == (int32_t)CH ? fi++ : pi++] = c;
		}
	}
	if (threadIdx.x == 0)
		s->nChunks = (int64_t)(nFull + nPart);
}

__global__ void __launch_bounds__(1024) kListScan(uint32_t* __restrict__ part,
                                                  uint32_t* __restrict__ listed)
{
	__shared__ unsigned long long lds[16];
	constexpr int per = kListWaves / 1024;
	uint32_t* p = part + per * threadIdx.x;
	unsigned long long sum = 0, total;
	for (int k = 0; k < per; k++)
		sum += p[k];
	uint32_t at = (uint32_t)scan1024(sum, lds, &total);
	for (int k = 0; k < per; k++)
	{
		const uint32_t q = p[k];
		p[k] = at;
		at += q;
	}
	if (threadIdx.x == 0)
		*listed = (uint32_t)total;
}

hipError_t launchLorList(const DCorr& c, int64_t n, uint32_t* part, uint32_t* list,
                         uint32_t* listed, hipStream_t st)
{
	kLorList<0><<<kListWaves / 4, 256, 0, st>>>(c, n, part, nullptr);
	kListScan<<<1, 1024, 0, st>>>(part, listed);
	kLorList<1><<<kListWaves / 4, 256, 0, st>>>(c, n, part, list);
	return hipGetLastError();
}

hipError_t launchStreamScan(const DPlan& pl, int64_t* tileOff, int nTiles, int64_t cap,
                            TileChunk* chunks, StreamState* s, hipStream_t st)
{
	kStreamScan<<<1, 1024, 0, st>>>(pl, tileOff, nTiles, cap, chunks, s);
	return hipGetLastError();
}

hipError_t launchTileBack(const KArgs& a, const DTiles& T, const DPlanRead& pl,
                          const float* v, float* y, int persistent, hipStream_t st)
{
	if (pl.nChunks <= 0 && pl.nChunksDev == nullptr)
		return hipSuccess;
	if (pl.vexp != nullptr && a.pr.type != 1 && T.shape != 2)
	{
		// the scale word is followed by the finished-workgroups counter and
		// the 256-bin exponent histogram
		int* ve = const_cast<int*>(pl.vexp);
		unsigned int* done = reinterpret_cast<unsigned int*>(ve) + 1;
		const int64_t n = a.L.n;
		const unsigned g = (unsigned)std::min<int64_t>(std::max<int64_t>((n + 2047) / 2048, 1), 1024);
		kVExpScale<<<g, 256, 0, st>>>(v, n, done + 1, done, ve);
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess)
			return e;
	}
	DPlanRead q = pl;
	unsigned grid;
	if (pl.nChunksDev != nullptr)
		grid = (unsigned)persistent;
	else if (persistent > 0 && pl.queue != nullptr)
		grid = (unsigned)std::min<int64_t>(persistent, pl.nChunks);
	else
	{
		q.queue = nullptr;
		grid = (unsigned)pl.nChunks;
	}
	if (a.pr.type == 1)
		tileBackKind<true>(a, T, q, v, y, grid, st);
	else
		tileBackKind<false>(a, T, q, v, y, grid, st);
	return hipGetLastError();
}

template <bool TOF, bool S64, bool BRICK>
static hipError_t ratioLpe(const KArgs& a, int lpe, int parts, dim3 g, dim3 b, float* v,
                           hipStream_t st)
{
	auto go = [&](auto lanes) {
		constexpr int N = decltype(lanes)::value;
		if constexpr (!S64)
			if (parts > 1)
			{
				kEmRatio<TOF, N, S64, BRICK, kRayParts, false><<<g, b, 0, st>>>(a, v);
				return;
			}
		if (a.list != nullptr)
			kEmRatio<TOF, N, S64, BRICK, 1, true><<<g, b, 0, st>>>(a, v);
		else
			kEmRatio<TOF, N, S64, BRICK, 1, false><<<g, b, 0, st>>>(a, v);
	};
	switch (lpe)
	{
	case 1:
		go(std::integral_constant<int, 1>{});
		break;
	case 2:
		go(std::integral_constant<int, 2>{});
		break;
	case 4:
		go(std::integral_constant<int, 4>{});
		break;
	case 8:
		go(std::integral_constant<int, 8>{});
		break;
	default:
		return hipErrorInvalidValue;
	}
	return hipGetLastError();
}

template <bool TOF, bool S64>
static hipError_t ratioT(const KArgs& a, int lpe, int parts, dim3 g, dim3 b, float* v,
                         hipStream_t st)
{
	if (a.pr.type == 1)
	{
		auto go = [&](auto k) { k<<<g, b, a.pr.psf.ldsBytes, st>>>(a, v); };
		auto lanes = [&](auto tab, auto brick) {
			constexpr bool T = decltype(tab)::value, B = decltype(brick)::value;
			if constexpr (T)
				if (a.list != nullptr)
				{
					lpe == 4 ? go(kEmRatioDD<TOF, S64, T, B, 4, true>)
					         : go(kEmRatioDD<TOF, S64, T, B, 1, true>);
					return;
				}
			lpe == 4 ? go(kEmRatioDD<TOF, S64, T, B, 4, false>)
			         : go(kEmRatioDD<TOF, S64, T, B, 1, false>);
		};
		using Y = std::true_type;
		using N = std::false_type;
		if (a.xb != nullptr)
			a.rays != nullptr ? lanes(Y{}, Y{}) : lanes(N{}, Y{});
		else
			a.rays != nullptr ? lanes(Y{}, N{}) : lanes(N{}, N{});
		return hipGetLastError();
	}
	return a.xb != nullptr ? ratioLpe<TOF, S64, true>(a, lpe, parts, g, b, v, st)
	                       : ratioLpe<TOF, S64, false>(a, lpe, parts, g, b, v, st);
}

// One workgroup per row of bricks (y, z), its threads along it: no division
// by the image's sizes in the loop.  5.1 M voxels 22 -> 13 us.
__global__ void __launch_bounds__(256)
    kToBricks(const float* __restrict__ x, float* __restrict__ xb, int nx, int ny, int nz,
              int64_t nvox, int64_t bvox)
{
	const int bnx = brickNx(nx), bny = brickNy(ny);
	const int by = (int)blockIdx.x % bny, bz = (int)blockIdx.x / bny;
	const float* src = x + (int64_t)blockIdx.y * nvox;
	float* dst = xb + (int64_t)blockIdx.y * bvox + (int64_t)blockIdx.x * bnx * 32;
	for (int o = (int)threadIdx.x; o < bnx * 32; o += 256)
	{
		const int w = o & 31;
		const int vx = (o >> 5) * 4 + (w & 3), vy = by * 4 + ((w >> 2) & 3), vz = bz * 2 + (w >> 4);
		dst[o] = (vx < nx && vy < ny && vz < nz) ? src[((int64_t)vz * ny + vy) * nx + vx] : 0.f;
	}
}

hipError_t launchToBricks(const DImage& im, const float* x, float* xb, hipStream_t st)
{
	const int64_t bvox = brickFrameVoxels(im.nx, im.ny, im.nz);
	const unsigned rows = (unsigned)(brickNy(im.ny) * brickNz(im.nz));
	for (int64_t f = 0; f < im.nt; f += 65535)
		kToBricks<<<dim3(rows, (unsigned)std::min<int64_t>(65535, im.nt - f)), 256, 0, st>>>(
		    x + f * im.nvox, xb + f * bvox, im.nx, im.ny, im.nz, im.nvox, bvox);
	return hipGetLastError();
}

hipError_t launchEmRatio(const KArgs& a, int lpe, float* v, hipStream_t st, int block,
                         int64_t grid)
{
	if (a.xb != nullptr && a.bvox != brickFrameVoxels(a.im.nx, a.im.ny, a.im.nz))
		return hipErrorInvalidValue;
	if (a.pr.type == 1)
		lpe = a.L.n <= kDDLanesUpTo ? 4 : 1;
	if (a.list != nullptr && a.pr.type == 1 && a.rays == nullptr)
		return hipErrorInvalidValue;
	const int parts = a.pr.type == 0 && !a.pr.setup64 && a.list == nullptr &&
	                          a.L.n * (int64_t)a.pr.numRays <= kSplitRays
	                      ? kRayParts
	                      : 1;
	const int64_t threads = a.L.n * lpe * parts;
	int64_t nb = grid > 0 ? grid : (threads + block - 1) / block;
	if (nb > 0x7ffffff0)
		nb = 0x7ffffff0;
	nb = (nb + kXcds - 1) / kXcds * kXcds;  // xcdRange is a bijection on [0, nb)
	if (nb < kXcds)
		nb = kXcds;
	const dim3 g((unsigned)nb), b((unsigned)block);
	const bool tof = a.pr.useTof != 0;
	if (a.pr.setup64)
		return tof ? ratioT<true, true>(a, lpe, parts, g, b, v, st)
		           : ratioT<false, true>(a, lpe, parts, g, b, v, st);
	return tof ? ratioT<true, false>(a, lpe, parts, g, b, v, st)
	           : ratioT<false, false>(a, lpe, parts, g, b, v, st);
}

hipError_t launchSensValue(const KArgs& a, float* v, hipStream_t st)
{
	int64_t nb = (a.L.n + 255) / 256;
	if (nb > 0x7ffffff0)
		nb = 0x7ffffff0;
	nb = (nb + kXcds - 1) / kXcds * kXcds;  // xcdRange is a bijection on [0, nb)
	const unsigned g = (unsigned)std::max<int64_t>(nb, kXcds);
	if (a.pr.setup64)
		a.xb ? kSensValue<true, true><<<g, 256, 0, st>>>(a, v)
		     : kSensValue<true, false><<<g, 256, 0, st>>>(a, v);
	else
		a.xb ? kSensValue<false, true><<<g, 256, 0, st>>>(a, v)
		     : kSensValue<false, false><<<g, 256, 0, st>>>(a, v);
	return hipGetLastError();
}

}  // namespace yrtmi
