// Tile plans: Siddon walks and distance-driven footprints binned by image
// tile, and the kernels that build and use them (host-side launchers).
#pragma once

#include "yrtmi_rays.hpp"

#include <algorithm>

namespace yrtmi
{

// Image tiles held in LDS by one workgroup, by shape (64-bit fixed-point
// voxels, DD FP64, FP32 for shape 2):
//   0: 16 x 16 x 16 (32 KB, 256 threads)   1: 32 x 32 x 16 (128 KB, 512)
//   2: 32 x 32 x 32 (128 KB FP32, 1024)    3: 32 x 32 x 8 (64 KB, 512)
constexpr int kNumTileShapes = 4;
__host__ __device__ constexpr int tileDim(int shape, int axis)
{
	return shape == 0 ? 16 : (shape == 2 ? 32 : (axis < 2 ? 32 : (shape == 1 ? 16 : 8)));
}
__host__ __device__ constexpr int tileThreads(int shape)
{
	return shape == 0 ? 256 : (shape == 2 ? 1024 : 512);
}
// Binning keeps a counter (count pass) and a counter plus a 32-bit base
// (fill pass; a plan holds fewer than 2^32 records) per (tile, length
// class) in LDS; length classes are added while tiles x classes <= kMaxBins
// and the device's LDS per workgroup holds them.
constexpr int kMaxBins = 16384;
constexpr int kMaxClasses = 16;
// Threads of a binning workgroup, which share its LDS counters (64 KB in the
// fill pass with 8192 bins: two workgroups per CU, 16 waves of 512 threads).
// Fill pass of 8.4 M LORs x 4 rays: 256 threads 4.2 ms, 512 2.9, 1024 4.7.
constexpr int kBinThreads = 512;

// Entry record of a ray in a tile: voxel within the tile (5 bits per axis),
// the ray's plane shift per axis (sidPlaneShift, 4 bits each, offset 8) and
// whether the tile is where the ray's walk starts (bit 31).
constexpr int kMaxShift = 7;
__host__ __device__ inline uint32_t packEntry(int lx, int ly, int lz, int dx, int dy,
                                              int dz, bool first)
{
	return (uint32_t)lx | ((uint32_t)ly << 5) | ((uint32_t)lz << 10) |
	       ((uint32_t)(dx + 8) << 15) | ((uint32_t)(dy + 8) << 19) |
	       ((uint32_t)(dz + 8) << 23) | (first ? 0x80000000u : 0u);
}

// A record's fine length class (0 .. 15), kept in entry-word bits that
// the record's fields leave free (Siddon: 27..30, packEntry; DD: 12..15,
// above the slice range) for the plan's per-chunk sort (kChunkSort).
// Siddon: its segments in the tile in 16 equal steps of the most a tile
// piece can hold (tx + ty + tz); DD: its footprint voxels per slice.
__host__ __device__ inline uint32_t withFineClass(bool dd, uint32_t pv, int segs, int L)
{
	if (dd)
	{
		const int ns = (int)((pv >> 6) & 63u) - (int)(pv & 63u) + 1;
		const int c = std::min(15, std::max(0, (segs + ns - 1) / std::max(ns, 1)));
		return pv | ((uint32_t)c << 12);
	}
	const int c = std::min(15, std::max(0, segs * 16 / std::max(L, 1)));
	return pv | ((uint32_t)c << 27);
}

// Words per plan record: Siddon key, alpha, entry; DD key, entry.
__host__ __device__ constexpr int recWords(bool dd) { return dd ? 2 : 3; }

__host__ __device__ inline int fineClassOf(bool dd, uint32_t pv)
{
	return (int)((pv >> (dd ? 12 : 27)) & 15u);
}

// Tiles of an image with nt frames: ntx * nty * ntz per frame, numbered
// ((f * ntz + tz) * nty + ty) * ntx + tx; tiles of tx * ty * tz voxels.
struct DTiles
{
	int32_t ntx, nty, ntz, nTiles;
	int32_t tx, ty, tz, shape;
	int32_t lx, ly, lz;  // log2 of tx, ty, tz (tile sides are powers of two)
};

// A chunk of one tile's records, processed by one workgroup.
struct TileChunk
{
	int64_t begin;
	int32_t tile;
	int32_t count;
};

// Records per chunk of a plan of `total` records: up to 4096, which amortise
// clearing and flushing the tile, and fewer when they would leave the chip
// idle (below 1024 chunks), down to one record per thread of a 16^3 tile's
// workgroup.  3000 events of one ray on 9 tiles: kTileBack 30 -> 10 us.
__host__ __device__ inline int chunkRecords(int64_t total)
{
	const int64_t c = (total / 1024 + 255) / 256 * 256;
	return (int)(c < 256 ? 256 : (c > 4096 ? 4096 : c));
}

// Plan being built.  Records are binned by (tile, length class): a record's
// class counts the cuts at or below its number of segments in the tile (DD:
// its footprint voxels in the tile), and
// within a tile the records are stored class by class, so that the lanes of
// a wave walk pieces of similar length.  Bin b = tile * C + class.
struct DPlan
{
	int32_t R;                  // rays per LOR
	int32_t C;                  // length classes (1 .. kMaxClasses)
	int32_t cut[kMaxClasses - 1];  // class k starts at cut[k-1] segments
	unsigned long long* count;  // [nTiles * C] records per bin (count pass)
	unsigned int* blockCnt;     // [grid][nTiles * C] records per workgroup and bin
	unsigned int* cursor;       // [nTiles * C] fill cursor within the bin
	const int64_t* tileOff;     // [nTiles * C] first record of the bin
	// records of recWords(DD) words: the key (lor * R + ray; DD: lor), the
	// alpha where the walk enters the tile (Siddon, its bits), the entry
	// word (packEntry; DD: the record's slices in the slab, binRayDD) with
	// its fine length class
	uint32_t* rec;
	const float4* ray;          // ray table (rayEntry + sidStore / ddStore, kRayPrep)
	int* err;                   // set when a tile range would overflow
	const int* skip;            // (nullable) the fill pass does nothing if set
	const uint32_t* listed;     // (nullable) LORs there are, as KArgs::listed
	int64_t listFirst;
};

// Cuts of a plan's length classes (DPlan::cut) for its number of classes.
// Siddon: at fractions of the longest piece a tile can hold (tx + ty + tz
// segments); DD: at multiples of the slices of a tile slab (a piece of a
// footprint a few voxels wide and high holds a few voxels per slice; 16
// classes are about 15 % apart where most pieces lie).
inline void lengthCuts(DPlan& pl, bool dd, const DTiles& T)
{
	static const int d16[15] = {1, 2, 3, 4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40},
	                 d8[7] = {1, 2, 4, 8, 12, 16, 24}, d4[3] = {2, 6, 16}, d2[1] = {8};
	static const int s8[7] = {3, 6, 9, 12, 16, 21, 28}, s4[3] = {6, 12, 21}, s2[1] = {12};
	const int* f = dd ? (pl.C == 16 ? d16 : (pl.C == 8 ? d8 : (pl.C == 4 ? d4 : d2)))
	                  : (pl.C == 8 ? s8 : (pl.C == 4 ? s4 : s2));
	const int L = dd ? std::max(T.tx, T.ty) : T.tx + T.ty + T.tz;
	for (int k = 0; k < pl.C - 1; k++)
		pl.cut[k] = std::max(1, L * f[k] / (dd ? 4 : 40));
}

// Tiles of shape `shape` of an image of nt frames (nTiles 0: 2^31 or more).
inline DTiles tilesOf(int shape, int64_t nx, int64_t ny, int64_t nz, int64_t nt)
{
	DTiles T{};
	T.shape = shape;
	T.tx = tileDim(shape, 0);
	T.ty = tileDim(shape, 1);
	T.tz = tileDim(shape, 2);
	T.lx = __builtin_ctz((unsigned)T.tx);
	T.ly = __builtin_ctz((unsigned)T.ty);
	T.lz = __builtin_ctz((unsigned)T.tz);
	T.ntx = (int32_t)((nx + T.tx - 1) / T.tx);
	T.nty = (int32_t)((ny + T.ty - 1) / T.ty);
	T.ntz = (int32_t)((nz + T.tz - 1) / T.tz);
	const int64_t n = (int64_t)T.ntx * T.nty * T.ntz * nt;
	T.nTiles = n < (int64_t(1) << 31) ? (int32_t)n : 0;
	return T;
}

// Room for the records of one DD footprint that calls without a plan leave, on
// the average of a batch.  An interval of l voxels at any offset meets 1 + l / T
// tiles of T on average: in each slab of tiles along the major axis the
// footprint's minor range, its width (crystal, PSF extent ext) and what the line
// moves across the slab, at most a slab's length; axially its height, and over
// all slabs what the line rises, at most the image.  8 per slab at least, up to 128
// (footprints of a few voxels: mostly below 4).
inline int64_t ddRecordsPerLor(const DTiles& T, float vx, float vy, float vz, float tt, float tz,
                               float ext)
{
	const double slabs = std::max(T.ntx, T.nty), vMin = std::min(vx, vy), vMax = std::max(vx, vy);
	const double minor = 1.0 + vMax / vMin + (1.5 * tt + 2.0 * ext) / vMin / T.tx;
	const double r = minor * (slabs * (1.0 + (double)tz / vz / T.tz) + T.ntz);
	return std::max((int64_t)std::min(128.0, 8.0 * slabs), (int64_t)std::min(r + 1.0, 1e9));
}
// More than this: the direct kernel.
constexpr int64_t kStreamRecords = 512;

// Ray table of a Siddon plan, rayTabVec(S64) float4 per (LOR, ray) t = lor *
// R + ray.  The first two: the ray's end points after multi-ray offsets,
// motion and the image offset (q1, q2, exactly as the walk sets it up) and
// two words.  FP64 set-up: its TOF value and its frame (-1: skipped).  FP32
// set-up: the walk's first voxel (10 bits per axis) and its frame with the
// plane shifts (rayWord); two more float4 hold the ray's set-up (sidStore),
// from which it is cut into its tiles (sidPieces) and walks re-entered at a
// tile record start without redoing it.
constexpr int rayTabVec(bool S64)
{
	return S64 ? 2 : 4;
}

__device__ __forceinline__ void rayEntry(float4* tab, int vec, uint32_t t, float3 q1, float3 q2,
                                         float w0, int32_t w1)
{
	tab[vec * (uint64_t)t] = make_float4(q1.x, q1.y, q1.z, q2.x);
	tab[vec * (uint64_t)t + 1] = make_float4(q2.y, q2.z, w0, __int_as_float(w1));
}

// Frame (below 65535: a plan has fewer tiles) and plane shifts of an FP32
// entry; a ray that is skipped, or misses the image, has the frame 0xffff.
constexpr uint32_t kNoFrame = 0xffffu;
__device__ __forceinline__ uint32_t rayWord(int frame, int dx, int dy, int dz)
{
	return (uint32_t)frame | ((uint32_t)(dx + 8) << 16) | ((uint32_t)(dy + 8) << 20) |
	       ((uint32_t)(dz + 8) << 24);
}

// Plan in use.  queue != null: persistent launch, workgroups take chunks
// from queue[0] (queue[1] counts finished workgroups; the last one resets
// both, so the next launch starts from zero without a memset).
struct DPlanRead
{
	int32_t R;
	const TileChunk* chunks;
	int64_t nChunks;
	const uint32_t* rec;  // records, recWords(DD) words each (DPlan::rec)
	const float4* ray;    // rayEntry + sidStore (Siddon) or ddStore (DD) table
	unsigned int* queue;
	// binade E of the median nonzero |v| of the launch (kVExpScale
	// before each launch): sets the fixed-point scale of the tile
	// accumulation
	const int* vexp;
	// plans made and used on the device (launchStreamScan): the chunk count,
	// and an error word that, when set, leaves the image untouched
	const int64_t* nChunksDev;
	const int* err;
};

// State of a plan made on the device: cleared before each batch, together
// with the bins' counts and cursors behind it.
struct StreamState
{
	int64_t nChunks;
	int err;  // 1 / 2: as DPlan::err; 4: more records than there is room for
	int pad;
	unsigned int queue[260];  // as a plan's queue words
};
// Clears `words` 32-bit words.
hipError_t launchClearWords(unsigned int* p, int64_t words, hipStream_t st);
// list = the elements below n (> 0) of the LORs that an EM subset with these
// corrections does not skip, in order; *listed, their number; part, kListWaves
// words of scratch.
constexpr int kListWaves = 4096;
hipError_t launchLorList(const DCorr& c, int64_t n, uint32_t* part, uint32_t* list,
                         uint32_t* listed, hipStream_t st);
// From pl.count: pl.tileOff, the chunk table (chunkRecords of the total,
// full chunks first) and s->nChunks; s->err |= 4 and no chunks when there
// are more than `cap` records or an error before.  One workgroup.
hipError_t launchStreamScan(const DPlan& pl, int64_t* tileOff, int nTiles, int64_t cap,
                            TileChunk* chunks, StreamState* s, hipStream_t st);

// LORs up to which a DD forward takes four lanes per LOR (3 waves for each of
// the chip's 1024 SIMDs at one).  96 x 96 x 48, four lanes against one: 65536
// LORs 94 / 172 us, 196608 205 / 212, 262144 260 / 254; 200 x 200 x 128 TOF:
// 116 / 220, 252 / 302, 336 / 425.
constexpr int64_t kDDLanesUpTo = 196608;

// Rays up to which a Siddon forward takes kRayParts lanes per ray (FP32 set-up):
// a walk is a chain of steps and gathers, and these fill 4 waves for each of the
// chip's SIMDs at most.  One lane against four, us: 4096 rays of 200 x 200 x 128
// 65 / 23 (TOF 22 / 12), 65536 77 / 47 (36 / 31), 98304 78 / 76 (39 / 48); of 96 x
// 96 x 48 27 / 12, 23 / 20, 28 / 28.
constexpr int kRayParts = 4;
constexpr int64_t kSplitRays = 65536;

// LDS of the fill pass: an int counter and a 32-bit base per bin.
inline size_t binLdsBytes(int nB)
{
	return (size_t)nB * (sizeof(int) + sizeof(uint32_t));
}
// The plan's ray table for a.L (before the binning passes).
// *err |= 2 for a ray whose plane shift is out of a record's range.
hipError_t launchRayPrep(const KArgs& a, float4* tab, int* err, hipStream_t st);
// pass 0: count; pass 1: fill (same grid in both).
hipError_t launchBin(int pass, const KArgs& a, const DTiles& T, const DPlan& pl,
                     int grid, hipStream_t st);
// Each chunk's records (nChunks chunks, device table) ordered by their fine
// length class, in place (kChunkSort).
hipError_t launchChunkSort(bool dd, const DPlan& pl, const TileChunk* chunks, int64_t nChunks,
                           hipStream_t st);
// y += backprojection of v (per LOR) through the plan's records: one
// workgroup per chunk, or `persistent` workgroups on the chunk queue.
hipError_t launchTileBack(const KArgs& a, const DTiles& T, const DPlanRead& pl,
                          const float* v, float* y, int persistent, hipStream_t st);
// Whether forward projections of n LORs of `rays` rays (DD: one) gather from the
// image's bricked copy.  A brick's line serves segments of a ray that rows split
// over lines; the four lanes of a LOR's rays side by side share rows' lines as
// well, and the bricked Siddon walk has a quarter more instructions.  So four rays
// per LOR and more take bricks where an XCD's 4 MB L2 holds less than half of a
// frame (LORs in locality order read one frame at a time), fewer rays and DD from small
// images on, where the call is long enough for the copy (its launch, and 3 ps a
// voxel).  Rows / bricks, us, EM ratios of list-mode events of a phantom, in
// locality order and as acquired:
//   2 M LORs of  96 x 96 x 48            128 x 128 x 96           4 M: 200 x 200 x 128
//   1 ray        491 / 399  903 / 856    870 / 761  1468 / 1329  3030 / 2603  7682 / 5340
//   1 ray, TOF   308 / 296  500 / 483    520 / 498   766 / 717   1564 / 1497  3026 / 2333
//   3 rays, TOF  629 / 613  903 / 800   1088 / 950  1527 / 1347
//   4 rays       968 / 1008 1100 / 1132 1462 / 1503 2284 / 1875  5177 / 4712  9923 / 6773
//   4 rays, TOF  530 / 620  583 / 663    784 / 826  1077 / 974   2358 / 2210  3810 / 2842
//   DD          1222 / 1295 2128 / 1796 2566 / 2055 5363 / 3717
//   DD, TOF      828 / 698  1146 / 930  1997 / 1479 2530 / 1896
// 4 rays at 128^3: 1479 / 1487 and 2152 / 1820 with TOF, 3067 / 3069 and 5535 / 4147
// without; 8 frames of 128 x 128 x 64 1239 / 1369, 1401 / 1481.  Fewer LORs of 96 x
// 96 x 48, TOF, in order: 1 ray 250 k 54 / 61, 500 k 95 / 101, 1 M 171 / 169; 3 rays
// 125 k 51 / 61, 250 k 102 / 104; DD 125 k 70 / 70; of 64^3, 1 ray, 500 k 70 / 69.
// (A frame's bricks are indexed in 32 bits, padding included, which a frame
// of few voxels along one axis, or of just below 2^31, may exceed.)
constexpr int64_t kBrickVoxels = int64_t(1) << 21;
inline bool useBricks(int64_t nx, int64_t ny, int64_t nz, int64_t frames, bool dd, int rays,
                      int64_t n)
{
	if (brickFrameVoxels((int)nx, (int)ny, (int)nz) >= (int64_t(1) << 31))
		return false;
	const int64_t frame = nx * ny * nz, all = frame * frames;
	if (!dd && rays >= 4)
		return frame >= kBrickVoxels;
	return all >= kBrickVoxels || (dd ? all >= (1 << 20) && n >= (1 << 17)
	                                  : all >= (1 << 18) && n * rays >= (1 << 19));
}
// xb (nt frames of brickFrameVoxels floats) = bricked copy of x (nt frames
// of the image's voxels), padding voxels 0.
hipError_t launchToBricks(const DImage& im, const float* x, float* xb, hipStream_t st);
// v[e] = EM ratio of LOR e (0 where skipped), or with a.plain its projection,
// Siddon or DD (a.pr.type); Siddon reads a.xb (launchToBricks of a.x) where
// it is given, else a.x.  block threads (64 to 256, full waves) and grid
// workgroups (0: from the LORs), the latter rounded up to a multiple of 8.
hipError_t launchEmRatio(const KArgs& a, int lpe, float* v, hipStream_t st, int block = 256,
                         int64_t grid = 0);
// v[e] = sensitivity value of LOR e (factor x attenuation).
hipError_t launchSensValue(const KArgs& a, float* v, hipStream_t st);

}  // namespace yrtmi
