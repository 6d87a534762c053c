// gfx950 kernels of the polygon path: projection, triangle setup and clipping, ordered tile
// binning and the tile raster/shade kernel that reproduces the reference's fill loops.
//
// Reference files (relative to its Source/ folder): model projection modelAPI.cpp:214-281,
// setup and clipping renderCore.cpp:172-341, row intervals ITriangle2D.cpp:70-176, weight
// planes ITriangle2D.cpp:182-300, the 2x2 filler shader/fillerTemplates.h:92-385, shading
// shader/RgbaMultiply.h:74-175.
#include "pipeline.h"
#include "occlusion.h"

#include <type_traits>

namespace dfpsr {

// ---------------------------------------------------------------------------------------
// Projection of a task's point (modelAPI.cpp:237-242): a model point transformed to the world,
// to the camera and onto the screen; a camera-space corner projected; or the caller's
// ProjectedPoint as it is.  The setup projects the corners of each fan triangle it reads, so
// no pass over the points comes before it.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ Projected projectedPoint(const TaskDev &t, int32_t local) {
	if (t.pointKind == POINTS_PROJECTED) return reinterpret_cast<const Projected *>(t.points)[local];
	const f3 p = make3(t.points[local * 3], t.points[local * 3 + 1], t.points[local * 3 + 2]);
	if (t.pointKind == POINTS_CAMERA_SPACE) return cameraToScreen(t.camera, p);
	return cameraToScreen(t.camera, worldToCamera(t.camera.location, transformPoint(transformFrom(t.transform), p)));
}

// ---------------------------------------------------------------------------------------
// Triangle setup: renderTriangleFromData -> renderTriangleWithShader -> drawClippedTriangle
// -> drawSubTriangle (renderCore.cpp:220-341), one thread per fan triangle.
// ---------------------------------------------------------------------------------------
// n / d for 0 <= n < 2^24 and d >= 1 with a quotient below 2^21 (a command's pair index over
// its tile columns: at most a canvas's tiles, and its tile rows): both operands are exact in
// float and the float quotient is within one of the integer one, which one step corrects -- no
// integer division sequence.
__device__ __forceinline__ int32_t divSmall(int32_t n, int32_t d) {
	int32_t q = (int32_t)((float)n * __builtin_amdgcn_rcpf((float)d));
	if (q * d > n) q--;
	else if ((q + 1) * d <= n) q++;
	return q;
}

// (command, tile) pairs and newly used tiles counted by one thread of the setup kernel.
struct BinTally { int32_t pairs, tiles; };

// A command's tiles as the setup block bins them: the first tile and its column and row on the
// canvas, the width of the tile rectangle, the canvas's tiles per row, the command's first pair in
// the block's pairs, and whether its canvas is dense (pairCovers).
struct BinJob { int32_t index, firstTile, width, tilesX, pairStart, tileX, tileY, dense; };

// The job that pair p of the block belongs to: the last one that starts at or before it.
__device__ __forceinline__ int32_t jobOfPair(const BinJob *jobs, int32_t count, int32_t p) {
	int32_t lo = 0, hi = count - 1;
	while (lo < hi) {
		const int32_t mid = (lo + hi + 1) >> 1;
		if (jobs[mid].pairStart <= p) lo = mid; else hi = mid - 1;
	}
	return lo;
}

// Whether a command's rows can cover a pixel of the w x h tile whose first pixel is (x0, y0); asked
// for every (command, tile) pair of a dense canvas.  There most triangles are smaller than the pixel
// spacing and many cover no pixel centre, or none of a tile that their bound touches; a tile sorts,
// stages and walks every command it lists, so the longest lists bound the frame.  384 uneven jobs, without
// and with the test: 1 502 446 pairs and a longest list of 5 593, 1 311 070 and 2 029 (blocks that clip
// much bin without it); raster 2 006 and 823 us, setup 250 and 245.  96 views of 256x256: raster 388 and
// 294 us, setup 125 and 148.  Where triangles are larger the test does not pay: a 1080p terrain loses a
// quarter of its pairs, but its raster gains 2 us and its setup loses as much.
//
// A right edge ends row r at trunc(m / a), m = c - b * r (EdgeRows), so it keeps column x >= 1 exactly
// when m >= a * x, and column 0 when m > -a (truncation); a left edge starts it after trunc(m / a) and
// keeps column x >= 1 when m < a * x, column 0 when m <= -a.  m is linear in the row: if the best of
// the tile's first and last row fails at the tile's best column, the edge keeps nothing of the tile.
// What is left of few rows is decided by the rows themselves.
constexpr int32_t PAIR_EXACT_ROWS = 4;
__device__ __forceinline__ bool pairCovers(const TriangleRows &tr, int32_t x0, int32_t y0, int32_t w, int32_t h) {
	if (tr.flags & 64) return false;
	const int32_t left = tmax(x0, tr.clipL), right = tmin(x0 + w, tr.clipR);
	const int32_t top = tmax(y0, tr.alT), bottom = tmin(y0 + h, tr.alB);
	if (left >= right || top >= bottom) return false;
	if (tr.flags & 128) return true;
	bool missed = false;
#pragma unroll
	for (int k = 0; k < 3; k++) {
		const EdgeRows e = tr.edges[k];
		const int32_t kind = (tr.flags >> (2 * k)) & 3;
		const double first = __builtin_fma(-e.exact.b, (double)(top - tr.alT), e.exact.c);
		const double last = __builtin_fma(-e.exact.b, (double)(bottom - 1 - tr.alT), e.exact.c);
		const double least = fmin(first, last), most = fmax(first, last), a = (double)e.exact.a;
		if (kind == 1) missed = missed || (right > 1 ? least >= a * (right - 1) : least > -a);
		if (kind == 2) missed = missed || (left > 0 ? most < a * left : most <= -a);
		if (kind == 3) missed = missed || most < 0.0;
	}
	if (missed) return false;
	if (bottom - top > PAIR_EXACT_ROWS) return true;
	bool covered = false;
#pragma clang loop unroll(disable)
	for (int32_t y = top; y < bottom; y++) {
		const RowInterval row = triangleRow(tr, y);
		covered = covered || tmax(row.left, left) < tmin(row.right, right);
	}
	return covered;
}
constexpr int32_t BIN_JOBS = 512;  // commands a setup block bins together (more: each thread bins its own)
constexpr int32_t TILE_TABLE_LOG2 = 10, TILE_TABLE = 1 << TILE_TABLE_LOG2, TILE_TABLE_PROBES = 8;
static_assert(TILE_TABLE % SCAN_BLOCK == 0, "the tile table's entries split evenly over a setup block");

// Enters pair slot[k] of tile[k] into the tile's list (direct bins).
__device__ __forceinline__ void binPair(const FrameDev &f, int32_t tile, int32_t slot, int32_t index) {
	if (slot < f.binCapacity) {
		f.tileList[(size_t)tile * f.binCapacity + slot] = index;
	} else {
		atomicOr(&f.counters[2], 2);
		atomicMax(&f.counters[6], slot + 1);
	}
}

// Keeps pair record r (packed lists): the command's slot in the tile's list.
__device__ __forceinline__ void recordPair(const FrameDev &f, int32_t r, int32_t tile, int32_t slot, int32_t index) {
	if (r < f.pairCapacity) f.pairRecords[r] = PairRecord{tile, slot, index};
	else atomicOr(&f.counters[2], 2);
}

// The differentiable shader's inputs of a fan triangle of a task.
__device__ __forceinline__ DiffInputs diffInputs(const TaskDev &task, int32_t fan) {
	const FanRecord rec = task.fans[fan];
	int32_t poly = rec.polygonFan >> 1, k = rec.polygonFan & 1;
	const float *tc = task.texcoords + poly * 16;
	const int32_t ca = 0, cb = (1 + k) * 4, cc = (2 + k) * 4;
	DiffInputs d;
	d.u = make3(tc[ca], tc[cb], tc[cc]);
	d.v = make3(tc[ca + 1], tc[cb + 1], tc[cc + 1]);
	d.point[0] = rec.corner[0];
	d.point[1] = rec.corner[1];
	d.point[2] = rec.corner[2];
	return d;
}

// What the emit of a fan triangle needs of its task and canvas, read before the block's prefix sums
// (with scalar loads where the wavefront has one task), so that no load chain starts after them.
struct EmitTarget {
	int32_t local, canvas, flags;  // the fan triangle's index in its task; the canvas slot; Command::flags
	int32_t width, height, tileBase, tilesX, tilesY, dense;
};
__device__ __forceinline__ EmitTarget emitTarget(const FrameDev &f, int32_t g, int32_t ti) {
	const TaskDev &t = f.tasks[ti];
	const CanvasDev &cv = f.canvases[t.canvas];
	return EmitTarget{g - t.fanBase, t.canvas, (t.camera.perspective != 0 ? 0 : 1) | (t.filter != 0 ? 2 : 0),
	                  cv.width, cv.height, cv.tileBase, cv.tilesX, cv.tilesY, cv.dense};
}

// Writes draw command `index` with its row setup and enters it into every tile it can touch: the
// columns of cut(wholeBound, canvas), the rows of the aligned raster bound (ITriangle2D.cpp:70-84).
// With direct bins the index goes into the tile's list at once (in any order: the raster sorts each
// list); otherwise the tile's count grows here and a pair record (tile, slot, command) keeps the slot
// until the counts are scanned and the list is filled from the records.
__device__ void emitCommand(const FrameDev &f, int32_t index, const Command &cmd, const Projected *P, const EmitTarget &cv,
                            BinTally &tally, BinJob *jobs, int32_t jobBase) {
	f.commands[index] = cmd;
	const TriangleRows tr = triangleRows(P[0].flat, P[1].flat, P[2].flat, rectSides(0, 0, cv.width, cv.height));
	f.triangleRows[index] = tr;
	int32_t tx0 = 0, tx1 = -1, ty0 = 0, ty1 = -1;  // no tiles when the bound misses the canvas
	if (tr.clipR > tr.clipL) {
		// The columns and rows are at least 0 here, so shifts divide.
		tx0 = tr.clipL >> f.tileShiftW;
		tx1 = (tr.clipR - 1) >> f.tileShiftW;
		ty0 = tr.alT >> f.tileShiftH;
		ty1 = tmin((tr.alB - 2) >> f.tileShiftH, cv.tilesY - 1);
	}
	const int32_t w = tx1 - tx0 + 1, count = tmax(w, 0) * tmax(ty1 - ty0 + 1, 0);
	if (jobs) {
		// Binned later by the whole block, pairs spread over its threads.  Every command writes
		// its job, with no pairs when it touches no tile.
		jobs[index - jobBase] = BinJob{index, cv.tileBase + ty0 * cv.tilesX + tx0, tmax(w, 1), cv.tilesX, tally.pairs, tx0, ty0, cv.dense};
		tally.pairs += count;
		return;
	}
	if (f.binCapacity == 0) {
		// Packed lists, this thread alone: records reserved for the command's pairs at once.
		const int32_t recordBase = count > 0 ? atomicAdd(&f.counters[7], count) : 0;
		for (int32_t i = 0; i < count; i++) {
			const int32_t tile = cv.tileBase + (ty0 + i / w) * cv.tilesX + tx0 + i % w;
			recordPair(f, recordBase + i, tile, atomicAdd(&f.tileCount[tile], 1), index);
		}
		return;
	}
	// Direct bins of this thread alone: the slot atomics of up to eight tiles are in flight
	// together before their list entries are written.
	constexpr int32_t BATCH = 8;
	for (int32_t base = 0; base < count; base += BATCH) {
		int32_t tile[BATCH], slot[BATCH];
#pragma unroll
		for (int k = 0; k < BATCH; k++) {
			const int32_t i = base + k;
			tile[k] = i < count ? cv.tileBase + (ty0 + i / w) * cv.tilesX + tx0 + i % w : -1;
			slot[k] = tile[k] >= 0 ? atomicAdd(&f.tileCount[tile[k]], 1) : 0;
		}
#pragma unroll
		for (int k = 0; k < BATCH; k++) {
			if (tile[k] < 0) continue;
			binPair(f, tile[k], slot[k], index);
			tally.pairs++;
			tally.tiles += slot[k] == 0 ? 1 : 0;
		}
	}
}

// The finished shader inputs of fan triangle (poly, k) of a task (Shader.h:37-57,
// RgbaMultiply.h:37-58): corner colours and texture coordinates, texture slots, the shader
// variant flags.
__device__ ShaderInputs triangleShader(const TaskDev &t, int32_t poly, int32_t k) {
	const float *col = t.colors + poly * 16;
	const float *tc = t.texcoords + poly * 16;
	const int32_t ca = 0, cb = (1 + k) * 4, cc = (2 + k) * 4;
	ShaderInputs si;
	si.red = make3(col[ca], col[cb], col[cc]);
	si.green = make3(col[ca + 1], col[cb + 1], col[cc + 1]);
	si.blue = make3(col[ca + 2], col[cb + 2], col[cc + 2]);
	si.alpha = make3(col[ca + 3], col[cb + 3], col[cc + 3]);
	si.u1 = make3(tc[ca], tc[cb], tc[cc]);
	si.v1 = make3(tc[ca + 1], tc[cb + 1], tc[cc + 1]);
	si.u2 = make3(tc[ca + 2], tc[cb + 2], tc[cc + 2]);
	si.v2 = make3(tc[ca + 3], tc[cb + 3], tc[cc + 3]);
	int32_t part = t.polygonPart[poly];
	si.diffuse = t.partTexture[part * 2];
	si.light = t.partTexture[part * 2 + 1];
	finishShaderInputs(si);
	return si;
}

// The projected corners of fan triangle g (of task ti) and its polygon.
struct TriangleCorners {
	Projected P[3];
	int32_t poly, k;
};

__device__ __forceinline__ TriangleCorners loadCorners(const FrameDev &f, int32_t g, int32_t ti) {
	const TaskDev &t = f.tasks[ti];
	const FanRecord fan = t.fans[g - t.fanBase];
	TriangleCorners tc;
	tc.poly = fan.polygonFan >> 1;
	tc.k = fan.polygonFan & 1;
	for (int c = 0; c < 3; c++) tc.P[c] = projectedPoint(t, fan.corner[c]);
	return tc;
}

// The shading inputs of a fan triangle's draw commands, in the form of the frame's mode.
__device__ __forceinline__ void storeFanInputs(const FrameDev &f, int32_t index, int32_t ti, int32_t local, const TriangleCorners &tc) {
	if (f.mode == 0) f.shaders[index] = triangleShader(f.tasks[ti], tc.poly, tc.k);
	if (f.mode == 1) f.diffInputs[index] = diffInputs(f.tasks[ti], local);
}

__device__ __forceinline__ void loadInputs(ShaderInputs &in, const TaskDev &t, int32_t, const TriangleCorners &tc) { in = triangleShader(t, tc.poly, tc.k); }
__device__ __forceinline__ void loadInputs(DiffInputs &in, const TaskDev &t, int32_t local, const TriangleCorners &) { in = diffInputs(t, local); }
__device__ __forceinline__ void storeInputs(const FrameDev &f, int32_t index, const ShaderInputs &in) { f.shaders[index] = in; }
__device__ __forceinline__ void storeInputs(const FrameDev &f, int32_t index, const DiffInputs &in) { f.diffInputs[index] = in; }

// What setupTriangle does with the draw commands: count them, or lower the occlusion grid under
// their hulls (renderer_occludeFromExistingTriangles).
enum { SETUP_COUNT = 0, SETUP_OCCLUDE = 1 };

// occludeFromSortedHull of one Solid draw command's triangle (rendererAPI.cpp:218-239, with
// the triangle's wholeBound as the pixel bound, :246-258): every cell whose four corners are
// inside the triangle takes the larger corner depth if that is nearer.  The depth is +0 or
// more, whose float bits order as integers, so an integer atomic min keeps the nearest and
// leaves any negative cell value (sign bit set) in place, as the reference's '<' does.
__device__ void occludeFromCommand(const FrameDev &f, const Projected *P) {
	const Rect bound = triangleBound(P[0].flat, P[1].flat, P[2].flat);
	if (!hullCanOcclude(bound)) return;
	const float z[3] = {P[0].cs.z, P[1].cs.z, P[2].cs.z};
	const int bits = __float_as_int(hullDistance(z, 3));
	const l2 hull[3] = {P[0].flat, P[1].flat, P[2].flat};
	const Rect cells = outerCellBound(bound, f.gridW, f.gridH);
	for (int32_t cy = cells.t; cy < cells.bottom(); cy++)
		for (int32_t cx = cells.l; cx < cells.right(); cx++)
			if (cellInsideOfHull(hull, 3, cx, cy)) atomicMin(reinterpret_cast<int *>(f.occlusionGrid) + cy * f.gridW + cx, bits);
}

// Whether a command survives completeOcclusion (rendererAPI.cpp:190-215): always without a
// grid; otherwise when some cell under its bound is not nearer than its nearest corner.
__device__ __forceinline__ bool survivesOcclusion(const FrameDev &f, const Projected *P) {
	if (f.occlusionGrid == nullptr) return true;
	return commandVisibleInGrid(f.occlusionGrid, f.gridW, f.gridH, triangleBound(P[0].flat, P[1].flat, P[2].flat), P[0].cs.z,
	                            P[1].cs.z, P[2].cs.z);
}

// The draw commands of a fan triangle, counted or lowered into the occlusion grid.  clipPoly: the
// calling wavefront's clipped polygon in LDS.  Triangles that need clipping are rare; the lanes
// holding one take the wavefront's polygon in turn, so that the polygon (nine sub-vertices indexed
// at run time) lives in LDS instead of private scratch memory.  *single is set where the triangle
// makes one draw command, inside the clip frustum and front-facing.
template <int MODE>
__device__ __forceinline__ int32_t setupTriangle(const FrameDev &f, int32_t ti, const TriangleCorners &tc, ClipPolygon *clipPoly,
                                                 bool *single) {
	const TaskDev &t = f.tasks[ti];
	const CanvasDev &cv = f.canvases[t.canvas];
	if (cv.color == nullptr && cv.depth == nullptr) return 0;
	const Projected *P = tc.P;
	const CameraParams &cam = t.camera;
	if (triangleVisibility(P[0].cs, P[1].cs, P[2].cs, cam.cull) == VIS_HIDDEN) return 0;
	if (t.filter != 0) {
		const float *col = t.colors + tc.poly * 16;
		if (almostZero(col[3]) && almostZero(col[(1 + tc.k) * 4 + 3]) && almostZero(col[(2 + tc.k) * 4 + 3])) return 0;
	}
	if (triangleVisibility(P[0].cs, P[1].cs, P[2].cs, cam.clip) == VIS_FULL) {
		if (!frontFacing(P[0].flat, P[1].flat, P[2].flat)) return 0;
		if (MODE == SETUP_OCCLUDE) {
			if (t.filter == 0) occludeFromCommand(f, P);
			return 0;
		}
		if (!survivesOcclusion(f, P)) return 0;
		*single = true;
		return 1;
	}
	// The lanes here are exactly those that clip: one at a time, in lane order.
	int32_t count = 0;
	const uint64_t clipping = __ballot(1);
	const int32_t me = (int32_t)(threadIdx.x & 63);
	for (uint64_t pending = clipping; pending != 0; pending &= pending - 1) {
		if (me != __builtin_ctzll(pending)) continue;
		ClipPolygon &poly9 = *clipPoly;
		poly9.init(P[0].cs, P[1].cs, P[2].cs);
		for (int32_t s = 0; s < cam.clip.count; s++) poly9.clip(cam.clip.planes[s]);
		for (int32_t i = 0; i < poly9.count - 2; i++) {
			const SubVertex &va = poly9.v[0], &vb = poly9.v[1 + i], &vc = poly9.v[2 + i];
			Projected S[3] = {cameraToScreen(cam, va.cs), cameraToScreen(cam, vb.cs), cameraToScreen(cam, vc.cs)};
			if (!frontFacing(S[0].flat, S[1].flat, S[2].flat)) continue;
			if (MODE == SETUP_OCCLUDE) {
				if (t.filter == 0) occludeFromCommand(f, S);
				continue;
			}
			if (!survivesOcclusion(f, S)) continue;
			count++;
		}
	}
	return count;
}

// Writes the draw commands of a counted fan triangle from index offset on and bins them.  One round
// of the loop takes every lane of the wavefront whose triangle is single (its tests are not repeated),
// each further round one lane that clips: the code that makes a command is there once.
// The caller has stored the shading inputs of a single triangle, so that they hold no registers here;
// those of a clipped one are read again.
__device__ __forceinline__ void emitTriangle(const FrameDev &f, int32_t ti, const EmitTarget &target, TriangleCorners &tc, bool single,
                                             int32_t offset, BinTally &tally, ClipPolygon *clipPoly, BinJob *jobs,
                                             int32_t jobBase) {
	const CameraParams &cam = f.tasks[ti].camera;
	const bool perspective = (target.flags & 1) == 0;
	const int32_t me = (int32_t)(threadIdx.x & 63);
	uint64_t clipping = __ballot(!single);
	bool singles = true;
#pragma clang loop unroll(disable)
	while (singles || clipping != 0) {
		const bool mine = singles ? single : me == __builtin_ctzll(clipping);
		if (mine) {
			ClipPolygon &poly9 = *clipPoly;
			int32_t parts = 1, count = 0;
			if (!single) {
				poly9.init(tc.P[0].cs, tc.P[1].cs, tc.P[2].cs);
				for (int32_t s = 0; s < cam.clip.count; s++) poly9.clip(cam.clip.planes[s]);
				parts = poly9.count - 2;
			}
#pragma clang loop unroll(disable)
			for (int32_t i = 0; i < parts; i++) {
				Projected *S = tc.P;  // a clipped triangle's own corners are in its polygon
				f3 subB = make3(0.0f, 1.0f, 0.0f), subC = make3(0.0f, 0.0f, 1.0f);
				if (!single) {
					const SubVertex &va = poly9.v[0], &vb = poly9.v[1 + i], &vc = poly9.v[2 + i];
					S[0] = cameraToScreen(cam, va.cs);
					S[1] = cameraToScreen(cam, vb.cs);
					S[2] = cameraToScreen(cam, vc.cs);
					subB = make3(va.subB, vb.subB, vc.subB);
					subC = make3(va.subC, vb.subC, vc.subC);
					if (!frontFacing(S[0].flat, S[1].flat, S[2].flat) || !survivesOcclusion(f, S)) continue;
					storeFanInputs(f, offset + count, ti, target.local, tc);
				}
				Command c;
				const f2 is[3] = {S[0].is, S[1].is, S[2].is};
				c.plane = weightPlanes(is, make3(S[0].cs.z, S[1].cs.z, S[2].cs.z), subB, subC, perspective);
				c.task = ti; c.flags = target.flags;
				emitCommand(f, offset + count, c, S, target, tally, jobs, jobBase);
				count++;
			}
		}
		if (singles) singles = false;
		else clipping &= clipping - 1;
	}
}

// Exclusive prefix over one value per thread of an NT-thread workgroup (NT a multiple of 64);
// returns the total.  Each wavefront scans its 64 values with lane shuffles, then the
// wavefront totals meet in waveTotals[NT / 64]: two barriers in all.
template <int NT>
__device__ __forceinline__ int32_t workgroupPrefix(int32_t value, int32_t &before, int32_t *waveTotals) {
	const int32_t lane = (int32_t)(threadIdx.x & 63), wave = (int32_t)(threadIdx.x >> 6);
	int32_t x = value;
#pragma unroll
	for (int32_t offset = 1; offset < 64; offset <<= 1) {
		const int32_t y = __shfl_up(x, offset, 64);
		if (lane >= offset) x += y;
	}
	if (NT == 64) {
		__syncthreads();  // a barrier like the multi-wavefront form
		before = x - value;
		return __shfl(x, 63, 64);
	}
	if (lane == 63) waveTotals[wave] = x;
	__syncthreads();
	int32_t waveBase = 0, total = 0;
#pragma unroll
	for (int32_t w = 0; w < NT / 64; w++) {
		const int32_t v = waveTotals[w];
		waveBase += w < wave ? v : 0;
		total += v;
	}
	__syncthreads();  // waveTotals may be written again right after
	before = waveBase + x - value;
	return total;
}

// Block-wide exclusive scan of one int32 per thread of a SCAN_BLOCK-thread block; returns the
// block total.
__device__ int32_t blockExclusiveScan(int32_t value, int32_t &exclusive) {
	__shared__ int32_t waveTotals[SCAN_BLOCK / 64];
	return workgroupPrefix<SCAN_BLOCK>(value, exclusive, waveTotals);
}

// The task of fan triangle g.  A wavefront's triangles nearly always come from one task: its first
// triangle's task is searched with scalar loads, and where that task holds the last one too, it is
// every lane's (uniform).  Its fields -- camera planes, transform, array bases -- are then read with
// scalar loads as well, instead of one dependent vector load per field and lane: two frustums of six
// planes are twelve such loads in a row.
__device__ __forceinline__ int32_t taskOf(const FrameDev &f, int32_t g, bool &uniform) {
	const int32_t firstFan = __builtin_amdgcn_readfirstlane(g);
	const int32_t first = __builtin_amdgcn_readfirstlane(findSegment(f.taskFanEnd, f.taskCount, firstFan));
	uniform = tmin(firstFan + 63, f.fanTotal - 1) < f.taskFanEnd[first];
	return uniform ? first : findSegment(f.taskFanEnd, f.taskCount, g);
}

// A count of FAN_SINGLE is one command that needs no clipping and has passed every test.
constexpr int32_t FAN_SINGLE = -1;
__global__ void __launch_bounds__(SCAN_BLOCK) k_setup_count(FrameDev f) {
	__shared__ ClipPolygon clipPolys[SCAN_BLOCK / 64];
	int32_t g = blockIdx.x * SCAN_BLOCK + threadIdx.x;
	int32_t n = 0;
	bool single = false;
	if (g < f.fanTotal) {
		bool uniform;
		const int32_t ti = taskOf(f, g, uniform);
		ClipPolygon *poly = &clipPolys[threadIdx.x >> 6];
		if (uniform) {
			const int32_t task = __builtin_amdgcn_readfirstlane(ti);
			n = setupTriangle<SETUP_COUNT>(f, task, loadCorners(f, g, task), poly, &single);
		} else {
			n = setupTriangle<SETUP_COUNT>(f, ti, loadCorners(f, g, ti), poly, &single);
		}
		f.fanCount[g] = single ? FAN_SINGLE : n;
	}
	int32_t ex;
	int32_t total = blockExclusiveScan(n, ex);
	if (threadIdx.x == 0) f.blockSums[blockIdx.x] = total;
}

// Exclusive scan of the per-block sums by one workgroup; writes the grand total.  Each thread
// takes a run of PER consecutive sums per step, so a step covers SCAN_BLOCK * PER of them.
__global__ void k_scan_block_sums(int32_t *blockSums, int32_t blocks, int32_t *total) {
	constexpr int32_t PER = 16;
	__shared__ int32_t carry;
	if (threadIdx.x == 0) carry = 0;
	__syncthreads();
	for (int32_t base = 0; base < blocks; base += SCAN_BLOCK * PER) {
		const int32_t first = base + (int32_t)threadIdx.x * PER;
		int32_t v[PER], run = 0;
#pragma unroll
		for (int k = 0; k < PER; k++) {
			v[k] = first + k < blocks ? blockSums[first + k] : 0;
			run += v[k];
		}
		int32_t ex;
		const int32_t sum = blockExclusiveScan(run, ex);
		const int32_t c = carry;
		int32_t at = c + ex;
#pragma unroll
		for (int k = 0; k < PER; k++) {
			if (first + k < blocks) blockSums[first + k] = at;
			at += v[k];
		}
		__syncthreads();
		if (threadIdx.x == 0) carry = c + sum;
		__syncthreads();
	}
	if (threadIdx.x == 0) *total = carry;
}

// The same over int64 values.
__device__ long long blockExclusiveScan64(long long value, long long &exclusive) {
	__shared__ long long s[SCAN_BLOCK];
	int32_t tid = threadIdx.x;
	s[tid] = value;
	__syncthreads();
	for (int32_t offset = 1; offset < SCAN_BLOCK; offset <<= 1) {
		long long v = (tid >= offset) ? s[tid - offset] : 0;
		__syncthreads();
		s[tid] += v;
		__syncthreads();
	}
	long long inclusive = s[tid];
	long long total = s[SCAN_BLOCK - 1];
	__syncthreads();
	exclusive = inclusive - value;
	return total;
}

// Exclusive scan of int64 block sums by one workgroup; writes the two 32-bit halves of the
// grand total.
__global__ void k_scan_block_sums64(long long *blockSums, int32_t blocks, int32_t *totalLow, int32_t *totalHigh) {
	__shared__ long long carry;
	if (threadIdx.x == 0) carry = 0;
	__syncthreads();
	for (int32_t base = 0; base < blocks; base += SCAN_BLOCK) {
		int32_t i = base + threadIdx.x;
		long long v = (i < blocks) ? blockSums[i] : 0;
		long long ex;
		long long sum = blockExclusiveScan64(v, ex);
		long long c = carry;
		if (i < blocks) blockSums[i] = c + ex;
		__syncthreads();
		if (threadIdx.x == 0) carry = c + sum;
		__syncthreads();
	}
	if (threadIdx.x == 0) {
		*totalLow = (int32_t)(carry & 0xFFFFFFFFll);
		*totalHigh = (int32_t)(carry >> 32);
	}
}

// sumBlocks = 1: each block adds up the totals of the blocks before it (and the last block writes
// the command total) instead of reading offsets scanned by k_scan_block_sums.
// Writes the draw commands of one block of SCAN_BLOCK fan triangles.  Two-pass form (SINGLE =
// false): k_setup_count has stored each triangle's command count, and the commands take dense
// indices from the prefix over all blocks.  Single-pass form (SINGLE = true): the block counts
// its own commands and writes them from index blockIdx.x * blockCapacity on, so no block waits
// for another and no count kernel runs before; indices keep submission order but leave gaps
// (the raster only orders commands by index).  A block with more commands than blockCapacity
// writes nothing and reports its count, and the frame runs again with room for it.
template <bool SINGLE>
__device__ __forceinline__ void setupEmit(const FrameDev &f, int32_t sumBlocks) {
	__shared__ ClipPolygon clipPolys[SCAN_BLOCK / 64];
	__shared__ int32_t blockTally[2];
	__shared__ int32_t recordBaseLds;
	__shared__ BinJob jobs[BIN_JOBS];
	__shared__ int32_t tableTile[TILE_TABLE];
	__shared__ int32_t tableCount[TILE_TABLE];
	int32_t g = blockIdx.x * SCAN_BLOCK + threadIdx.x;
	for (int32_t e = threadIdx.x; e < TILE_TABLE; e += SCAN_BLOCK) {  // empty before the prefix sums' barriers
		tableTile[e] = -1;
		tableCount[e] = 0;
	}
	int32_t ti = 0;
	TriangleCorners corners;
	EmitTarget target;
	typename std::conditional<SINGLE, ShaderInputs, DiffInputs>::type inputs;  // one pass: RGBA8 frames, two: mostly differentiable ones
	int32_t n;
	bool single = false;  // counted as one unclipped, front-facing command
	if (SINGLE) {
		// The corners and the shader inputs of a triangle that makes commands stay in registers
		// from the count to the emit; the shader inputs' loads are issued before the block's
		// prefix sums, so that their latency overlaps them.
		n = 0;
		if (g < f.fanTotal) {
			bool uniform;
			ti = taskOf(f, g, uniform);
			ClipPolygon *poly = &clipPolys[threadIdx.x >> 6];
			if (uniform) {
				const int32_t task = __builtin_amdgcn_readfirstlane(ti);
				corners = loadCorners(f, g, task);
				target = emitTarget(f, g, task);
				n = setupTriangle<SETUP_COUNT>(f, task, corners, poly, &single);
				if (single && f.mode == 0) loadInputs(inputs, f.tasks[task], target.local, corners);
			} else {
				corners = loadCorners(f, g, ti);
				target = emitTarget(f, g, ti);
				n = setupTriangle<SETUP_COUNT>(f, ti, corners, poly, &single);
				if (single && f.mode == 0) loadInputs(inputs, f.tasks[ti], target.local, corners);
			}
		}
	} else {
		n = 0;
		if (g < f.fanTotal) {
			n = f.fanCount[g];
			single = n == FAN_SINGLE;
			if (single) n = 1;
			bool uniform;
			ti = taskOf(f, g, uniform);
			// Loaded before the block's prefix sums, so that the latency overlaps them.
			if (uniform) {
				const int32_t task = __builtin_amdgcn_readfirstlane(ti);
				target = emitTarget(f, g, task);
				if (n > 0) {
					corners = loadCorners(f, g, task);
					if (f.mode == 1) loadInputs(inputs, f.tasks[task], target.local, corners);
				}
			} else {
				target = emitTarget(f, g, ti);
				if (n > 0) {
					corners = loadCorners(f, g, ti);
					if (f.mode == 1) loadInputs(inputs, f.tasks[ti], target.local, corners);
				}
			}
		}
	}
	int32_t ex;
	const int32_t blockCommands = blockExclusiveScan(n, ex);
	if (threadIdx.x < 2) blockTally[threadIdx.x] = 0;
	int32_t jobBase;
	bool room;
	if (SINGLE) {
		jobBase = (int32_t)blockIdx.x * f.blockCapacity;
		room = blockCommands <= f.blockCapacity;
		if (threadIdx.x == 0 && blockCommands > 0) {
			atomicAdd(&f.counters[0], blockCommands);
			if (!room) {
				atomicOr(&f.counters[2], 1);
				atomicMax(&f.counters[8], blockCommands);
			}
		}
	} else {
		if (sumBlocks) {
			int32_t partial = 0, unusedPrefix;
			for (int32_t i = threadIdx.x; i < (int32_t)blockIdx.x; i += SCAN_BLOCK) partial += f.blockSums[i];
			jobBase = blockExclusiveScan(partial, unusedPrefix);
			if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) f.counters[0] = jobBase + blockCommands;
		} else {
			jobBase = f.blockSums[blockIdx.x];
		}
		room = jobBase + blockCommands <= f.commandCapacity;
	}
	// The block's commands are binned together (below) when they fit the table and the command
	// arrays (a block past the capacity leaves its jobs unwritten).
	const bool together = blockCommands <= BIN_JOBS && room;
	BinTally tally{0, 0};
	if (g < f.fanTotal) {
		const int32_t offset = jobBase + ex;
		// The commands of a canvas's tasks are consecutive, so the offset at the first fan
		// triangle of each task bounds its canvas's first command: one atomic per task.
		if (target.local == 0) atomicMin(&f.canvasCommandBase[target.canvas], offset);
		if (n > 0) {
			if (!SINGLE && offset + n > f.commandCapacity) atomicOr(&f.counters[2], 1);
			else if (room) {
				if (single) {
					if (f.mode == (SINGLE ? 0 : 1)) storeInputs(f, offset, inputs);
					else storeFanInputs(f, offset, ti, target.local, corners);
				}
				emitTriangle(f, ti, target, corners, single, offset, tally, &clipPolys[threadIdx.x >> 6], together ? jobs : nullptr, jobBase);
			}
		}
	}
	if (together) {
		// Pairs of the block's commands, one per thread and round: job j owns pairs
		// [pairStart, pairStart + width * height) in command order.  A command whose setup ran
		// out of room (capacity) wrote no job; then no command of the frame is drawn anyway.
		int32_t pairBase;
		const int32_t pairs = blockExclusiveScan(tally.pairs, pairBase);
		for (int32_t k = 0; k < n; k++) jobs[ex + k].pairStart += pairBase;
		if (threadIdx.x == 0 && f.binCapacity == 0) recordBaseLds = pairs > 0 ? atomicAdd(&f.counters[7], pairs) : 0;
		__syncthreads();
		const int32_t recordBase = recordBaseLds;
		const int32_t jobCount = blockCommands;
		BinTally binned{0, 0};
		// Rounds of up to UNROLL pairs per thread.  The pairs of a round that go to one tile take
		// their slots with one global atomic: each pair draws a rank from the tile's entry in an
		// LDS table (TILE_TABLE entries, open addressing), one thread per entry then adds the
		// tile's count to its global count, and the pair's slot is the returned base plus its
		// rank.  A pair that finds no entry takes its slot with a global atomic of its own.
		constexpr int32_t UNROLL = 4;
		for (int32_t round = 0; round < pairs; round += UNROLL * SCAN_BLOCK) {
			// The pairs of dense canvases that no row covers; in a loop of its own, so that the other
			// frames fetch none of its code.
			uint32_t missed = 0;
			if (f.denseAny) {
#pragma clang loop unroll(disable)
				for (int u = 0; u < UNROLL; u++) {
					const int32_t p = round + (int32_t)threadIdx.x + u * SCAN_BLOCK;
					if (p >= pairs) break;
					const BinJob &j = jobs[jobOfPair(jobs, jobCount, p)];
					if (!j.dense) continue;
					const int32_t i = p - j.pairStart, row = divSmall(i, j.width), column = i - row * j.width;
					if (!pairCovers(f.triangleRows[j.index], (j.tileX + column) << f.tileShiftW, (j.tileY + row) << f.tileShiftH, f.tileW, f.tileH))
						missed |= 1u << u;
				}
			}
			int32_t tile[UNROLL], slot[UNROLL], index[UNROLL], entry[UNROLL];
#pragma unroll
			for (int u = 0; u < UNROLL; u++) {
				slot[u] = 0;
				const int32_t p = round + (int32_t)threadIdx.x + u * SCAN_BLOCK;
				tile[u] = -1;
				entry[u] = -1;
				if (p < pairs) {
					const BinJob &j = jobs[jobOfPair(jobs, jobCount, p)];
					const int32_t i = p - j.pairStart;
					const int32_t row = divSmall(i, j.width);
					index[u] = j.index;
					if ((missed >> u) & 1u) continue;
					tile[u] = j.firstTile + row * j.tilesX + (i - row * j.width);
					const int32_t h = (int32_t)(((uint32_t)tile[u] * 2654435761u) >> (32 - TILE_TABLE_LOG2));
					for (int32_t q = 0; q < TILE_TABLE_PROBES; q++) {
						const int32_t e = (h + q) & (TILE_TABLE - 1);
						const int32_t old = atomicCAS(&tableTile[e], -1, tile[u]);
						if (old == -1 || old == tile[u]) {
							entry[u] = e;
							break;
						}
					}
					slot[u] = entry[u] >= 0 ? atomicAdd(&tableCount[entry[u]], 1) : atomicAdd(&f.tileCount[tile[u]], 1);
				}
			}
			__syncthreads();
			{
				// Every entry's global atomic is issued before any of the returned bases is used.
				constexpr int32_t PER = TILE_TABLE / SCAN_BLOCK;
				int32_t entryTile[PER], entryBase[PER];
#pragma unroll
				for (int q = 0; q < PER; q++) entryTile[q] = tableTile[(int32_t)threadIdx.x + q * SCAN_BLOCK];
#pragma unroll
				for (int q = 0; q < PER; q++)
					entryBase[q] = entryTile[q] >= 0 ? atomicAdd(&f.tileCount[entryTile[q]], tableCount[(int32_t)threadIdx.x + q * SCAN_BLOCK]) : 0;
#pragma unroll
				for (int q = 0; q < PER; q++)
					if (entryTile[q] >= 0) tableCount[(int32_t)threadIdx.x + q * SCAN_BLOCK] = entryBase[q];
			}
			__syncthreads();
#pragma unroll
			for (int u = 0; u < UNROLL; u++) {
				const int32_t p = round + (int32_t)threadIdx.x + u * SCAN_BLOCK;
				const int32_t s = entry[u] >= 0 ? tableCount[entry[u]] + slot[u] : slot[u];
				const bool kept = tile[u] >= 0;
				// The wavefront's totals, so that the block adds them up with one LDS atomic each.
				binned.pairs += __popcll(__ballot(kept));
				binned.tiles += __popcll(__ballot(kept && s == 0));
				if (f.binCapacity == 0) {
					if (p < pairs) recordPair(f, recordBase + p, tile[u], s, index[u]);  // tile -1: missed
				} else if (kept) {
					binPair(f, tile[u], s, index[u]);
				}
			}
			if (round + UNROLL * SCAN_BLOCK >= pairs) break;  // the last round: the table is not needed again
			__syncthreads();
			for (int32_t e = threadIdx.x; e < TILE_TABLE; e += SCAN_BLOCK) {
				tableTile[e] = -1;
				tableCount[e] = 0;
			}
			__syncthreads();
		}
		if ((threadIdx.x & 63) == 0) tally = binned;
		else tally = BinTally{0, 0};
	}
	// The pair and used-tile totals, one global atomic per block.
	__syncthreads();
	if (tally.pairs) atomicAdd(&blockTally[0], tally.pairs);
	if (tally.tiles) atomicAdd(&blockTally[1], tally.tiles);
	__syncthreads();
	if (threadIdx.x == 0 && blockTally[0]) atomicAdd(&f.counters[1], blockTally[0]);
	if (threadIdx.x == 1 && blockTally[1]) atomicAdd(&f.counters[3], blockTally[1]);
}

// Bound by the latency of its loads, prefixes and atomics, not by bytes: with commands made in one
// place, the task's fields read as scalars before the prefix and no test repeated by the second pass,
// one pass takes 18.2 us of a 1080p terrain (20.2 before), 25.4 at 4K (31.6), 246 for 384 uneven jobs
// (256); two passes 47 us for 8 views of 1280x720 (52) and 148 for 96 of 256x256 (199).  The second
// pass gains from a fourth wavefront per SIMD where the blocks take several rounds of the chip (96
// views: 115 us against 132 at three, for 28 B of scratch); the single pass does not (4K: 26.0 against
// 25.4, the jobs 251 against 246).
__global__ void __launch_bounds__(SCAN_BLOCK) __attribute__((amdgpu_waves_per_eu(4, 4))) k_setup_emit(FrameDev f, int32_t sumBlocks) { setupEmit<false>(f, sumBlocks); }
__global__ void __launch_bounds__(SCAN_BLOCK) k_setup_single(FrameDev f) { setupEmit<true>(f, 0); }

// ---------------------------------------------------------------------------------------
// Binning into screen tiles.  List slots come from atomics on the tile counts, so a list is
// in no particular order; the raster kernel sorts it by command index, which restores
// submission order per pixel.
// ---------------------------------------------------------------------------------------

// Tile offsets and the ordered queue of non-empty tiles come from one scan of
// (count | nonEmpty << 32); the block-local queue position waits in tileFill in between.
__global__ void k_scan_tiles_local(FrameDev f) {
	int32_t i = blockIdx.x * SCAN_BLOCK + threadIdx.x;
	int32_t v = (i < f.tileTotal) ? f.tileCount[i] : 0;
	long long ex;
	long long total = blockExclusiveScan64((long long)v | ((long long)(v > 0) << 32), ex);
	if (i < f.tileTotal) {
		f.tileOffset[i] = (int32_t)(ex & 0xFFFFFFFFll);
		f.tileFill[i] = (int32_t)(ex >> 32);
	}
	if (threadIdx.x == 0) ((long long *)f.blockSums)[blockIdx.x] = total;
}

__global__ void k_scan_tiles_add(FrameDev f) {
	int32_t i = blockIdx.x * SCAN_BLOCK + threadIdx.x;
	if (i < f.tileTotal) {
		const long long base = ((const long long *)f.blockSums)[blockIdx.x];
		f.tileOffset[i] += (int32_t)(base & 0xFFFFFFFFll);
		if (f.tileCount[i] > 0) f.tileQueue[(int32_t)(base >> 32) + f.tileFill[i]] = i;
	}
	if (i == f.tileTotal - 1) {
		int32_t end = f.tileOffset[i] + f.tileCount[i];
		f.tileOffset[f.tileTotal] = end;
		if (end > f.pairCapacity) atomicOr(&f.counters[2], 2);
	}
}

// The packed lists from the pair records: each command goes to its slot after its tile's offset.
__global__ void k_bin_fill(FrameDev f) {
	const int32_t r = blockIdx.x * blockDim.x + threadIdx.x;
	if (f.counters[2] || r >= f.counters[7] || r >= f.pairCapacity) return;
	const PairRecord rec = f.pairRecords[r];
	if (rec.tile < 0) return;  // the command's triangle misses the tile
	f.tileList[f.tileOffset[rec.tile] + rec.slot] = rec.command;
}

// The tiles that a persistent grid draws first (forEachQueuedTile): those with the longest lists from
// the front of longTiles on, long ones from its back, in any order within the two.
__global__ void __launch_bounds__(256) k_long_tiles(FrameDev f) {
	const int32_t tile = blockIdx.x * blockDim.x + threadIdx.x;
	const int32_t n = tile < f.tileTotal ? f.tileCount[tile] : 0;
	const uint64_t below = (1ull << (threadIdx.x & 63)) - 1ull;
#pragma unroll
	for (int k = 0; k < 2; k++) {
		const bool mine = k == 0 ? n > LONGEST_LIST : n > LONG_LIST && n <= LONGEST_LIST;
		const uint64_t lanes = __ballot(mine);
		if (lanes == 0) continue;
		int32_t at = 0;
		if ((int32_t)(threadIdx.x & 63) == __builtin_ctzll(lanes)) at = atomicAdd(&f.counters[LONG_TILES + k], __popcll(lanes));
		at = __shfl(at, __builtin_ctzll(lanes), 64) + __popcll(lanes & below);
		if (mine) f.longTiles[k == 0 ? at : f.tileTotal - 1 - at] = tile;
	}
}

// ---------------------------------------------------------------------------------------
// Tile raster / shade.
// ---------------------------------------------------------------------------------------

// Sort of n distinct ints in LDS by the workgroup's NL lanes (n <= TILE_SORT_CAP).  Up to 4 NL
// values are ranked (each lane counts the values smaller than each of its own and writes them
// to those places: two barriers); longer lists take a bitonic sort.
template <int NL>
__device__ void sortLds(int32_t *a, int32_t n) {
	if (n <= NL) {
		const int32_t i = (int32_t)threadIdx.x;
		const int32_t v = i < n ? a[i] : 0;
		int32_t rank = 0;
		for (int32_t j = 0; j < n; j++) rank += a[j] < v ? 1 : 0;
		__syncthreads();
		if (i < n) a[rank] = v;
		__syncthreads();
		return;
	}
	if (n <= 4 * NL) {
		const int32_t i = (int32_t)threadIdx.x;
		int32_t v[4], rank[4] = {0, 0, 0, 0};
		for (int k = 0; k < 4; k++) v[k] = i + k * NL < n ? a[i + k * NL] : 0x7FFFFFFF;
		for (int32_t j = 0; j < n; j++) {
			const int32_t aj = a[j];
			for (int k = 0; k < 4; k++) rank[k] += aj < v[k] ? 1 : 0;
		}
		__syncthreads();
		for (int k = 0; k < 4; k++)
			if (i + k * NL < n) a[rank[k]] = v[k];
		__syncthreads();
		return;
	}
	int32_t size = 1;
	while (size < n) size <<= 1;
	for (int32_t i = n + (int32_t)threadIdx.x; i < size; i += NL) a[i] = 0x7FFFFFFF;
	__syncthreads();
	for (int32_t k = 2; k <= size; k <<= 1) {
		for (int32_t j = k >> 1; j > 0; j >>= 1) {
			for (int32_t i = threadIdx.x; i < size; i += NL) {
				int32_t ixj = i ^ j;
				if (ixj > i) {
					int32_t x = a[i], y = a[ixj];
					bool up = (i & k) == 0;
					if ((x > y) == up) { a[i] = y; a[ixj] = x; }
				}
			}
			__syncthreads();
		}
	}
}

// The four pixels of a lane's quad, held in registers for the whole tile.  MODE 0 holds the
// RGBA8 colours of the reference's shaders; MODE 1 (differentiable) holds float RGBA and the
// visibility id (draw command * 4 + quad lane) of the last write.
template <int MODE> struct QuadPixels;
template <> struct QuadPixels<0> {
	uint32_t color[4];
	float depth[4];
	uint32_t colorDirty, depthDirty;
};
template <> struct QuadPixels<1> {
	float r[4], g[4], b[4], a[4];
	int32_t vis[4];
	float depth[4];
	uint32_t colorDirty, depthDirty;
};

template <typename T> __device__ __forceinline__ T pick4(const T *v, int s) {
	return s == 0 ? v[0] : (s == 1 ? v[1] : (s == 2 ? v[2] : v[3]));
}
template <typename T> __device__ __forceinline__ void put4(T *v, int s, T x) {
	if (s == 0) v[0] = x; else if (s == 1) v[1] = x; else if (s == 2) v[2] = x; else v[3] = x;
}

// One quad of one command: which lanes the command covers and their weight-plane values,
// stepped exactly as the reference's loops step them -- the row-pair logic of fillShapeSuper
// (fillerTemplates.h:246-385), the incremental stepping of fillRowSuper (:195-244) and the
// side clipping of clipPixels (:92-108).
struct QuadEval {
	float l0[4], l1[4], l2[4];  // depth (1/W or W) and the two depth-divided vertex weights per lane
	int slot[4];                // pixel written by each lane (a missing row aliases the other row)
	bool clip[4];
	bool clipSides;
};

// n steps of both rows' weights by d, one rounded addition at a time as the reference steps
// them (n <= 0: none).  Four steps per trip keep the loop control of lanes with different n
// off most steps; the additions and their order are the same.
__device__ __forceinline__ void stepPair(f3 &wU, f3 &wL, const f3 &d, int32_t n) {
	int32_t i = 0;
#pragma clang loop unroll(disable)
	for (; i + 4 <= n; i += 4) {
		wU = add3(wU, d); wL = add3(wL, d);
		wU = add3(wU, d); wL = add3(wL, d);
		wU = add3(wU, d); wL = add3(wL, d);
		wU = add3(wU, d); wL = add3(wL, d);
	}
#pragma clang loop unroll(disable)
	for (; i < n; i++) { wU = add3(wU, d); wL = add3(wL, d); }
}

// upper/lower: row intervals of rows py and py + 1 (py even).  Returns false when the command
// does not touch the quad at px (even).
__device__ __forceinline__ bool evalQuad(const Projection &cmd, RowInterval upper, RowInterval lower, int32_t px, int32_t py,
                                         int32_t canvasHeight, QuadEval &e) {
	int32_t outerStart = tmin(upper.left, lower.left);
	int32_t outerEnd = tmax(upper.right, lower.right);
	int32_t innerStart = tmax(upper.left, lower.left);
	int32_t innerEnd = tmin(upper.right, lower.right);
	int32_t outerBlockStart = (int32_t)((uint32_t)outerStart & ~1u);
	int32_t outerBlockEnd = (int32_t)(((uint32_t)outerEnd + 1u) & ~1u);
	int32_t innerBlockStart = (int32_t)(((uint32_t)innerStart + 1u) & ~1u);
	int32_t innerBlockEnd = (int32_t)((uint32_t)innerEnd & ~1u);
	if (py + 1 >= canvasHeight) lower.right = lower.left;  // the missing last row of an odd canvas
	bool hasTop = upper.right > upper.left;
	bool hasBottom = lower.right > lower.left;
	if (!(hasTop || hasBottom)) return false;
	if (px < outerBlockStart || px >= outerBlockEnd) return false;

	const f3 dx = cmd.dx;
	const f3 dx2 = scale3(dx, 2.0f);
	f3 wU = weightAtPixel(cmd, outerBlockStart, py);
	f3 wL = add3(wU, cmd.dy);
	const bool splitSpan = innerBlockEnd > innerBlockStart;
	const bool inner = splitSpan && px >= innerBlockStart && px < innerBlockEnd;  // unclipped inner span
	const bool right = splitSpan && px >= innerBlockEnd;                         // clipped, right of it
	// The lanes of a wavefront take the same steps in the same places whatever part of the
	// row pair their quads are in: the pair chain to the quad (left part) or to the inner
	// span's start; past the inner span, its whole length at once and the chain to the quad.
	stepPair(wU, wL, dx2, (((inner || right) ? innerBlockStart : px) - outerBlockStart) >> 1);
	if (right) {
		float quadCount = (float)((innerBlockEnd - innerBlockStart) / 2);
		wU = add3(wU, scale3(dx2, quadCount));
		wL = add3(wL, scale3(dx2, quadCount));
		stepPair(wU, wL, dx2, (px - innerBlockEnd) >> 1);
	}
	e.clipSides = !inner;
	e.l0[0] = wU.x; e.l0[1] = wU.x + dx.x; e.l0[2] = wL.x; e.l0[3] = wL.x + dx.x;
	e.l1[0] = wU.y; e.l1[1] = wU.y + dx.y; e.l1[2] = wL.y; e.l1[3] = wL.y + dx.y;
	e.l2[0] = wU.z; e.l2[1] = wU.z + dx.z; e.l2[2] = wL.z; e.l2[3] = wL.z + dx.z;
	if (inner) {
		// Inside the span the four lanes step on their own, a quad at a time.
		int32_t x = innerBlockStart;
#pragma clang loop unroll(disable)
		for (; x + 4 <= px; x += 4) {
			for (int l = 0; l < 4; l++) { e.l0[l] = e.l0[l] + dx2.x; e.l1[l] = e.l1[l] + dx2.y; e.l2[l] = e.l2[l] + dx2.z; }
			for (int l = 0; l < 4; l++) { e.l0[l] = e.l0[l] + dx2.x; e.l1[l] = e.l1[l] + dx2.y; e.l2[l] = e.l2[l] + dx2.z; }
		}
#pragma clang loop unroll(disable)
		for (; x < px; x += 2) {
			for (int l = 0; l < 4; l++) { e.l0[l] = e.l0[l] + dx2.x; e.l1[l] = e.l1[l] + dx2.y; e.l2[l] = e.l2[l] + dx2.z; }
		}
	}
	e.slot[0] = hasTop ? 0 : 2;
	e.slot[1] = hasTop ? 1 : 3;
	e.slot[2] = hasBottom ? 2 : 0;
	e.slot[3] = hasBottom ? 3 : 1;
	if (e.clipSides) {
		int32_t x2 = px + 1;
		e.clip[0] = px >= upper.left && px < upper.right;
		e.clip[1] = x2 >= upper.left && x2 < upper.right;
		e.clip[2] = px >= lower.left && px < lower.right;
		e.clip[3] = x2 >= lower.left && x2 < lower.right;
	} else {
		e.clip[0] = e.clip[1] = e.clip[2] = e.clip[3] = true;
	}
	return true;
}

__device__ __forceinline__ bool evalQuad(const Command &cmd, RowInterval upper, RowInterval lower, int32_t px, int32_t py,
                                         int32_t canvasHeight, QuadEval &e) {
	return evalQuad(cmd.plane, upper, lower, px, py, canvasHeight, e);
}

// Vertex weights of a lane (fillRowSuper, fillerTemplates.h:222-238): perspective divides the
// depth-divided weights by 1/W.
__device__ __forceinline__ void laneWeights(const QuadEval &e, int l, bool affine, float &wa, float &wb, float &wc) {
	if (affine) {
		wb = e.l1[l];
		wc = e.l2[l];
	} else {
		float w = refinedReciprocal(e.l0[l]);
		wb = e.l1[l] * w;
		wc = e.l2[l] * w;
	}
	wa = 1.0f - (wb + wc);
}

// Depth test of getVisibility (fillerTemplates.h:110-152).
template <int MODE>
__device__ __forceinline__ bool quadVisibility(const QuadEval &e, const QuadPixels<MODE> &q, bool depthRead, bool affine, bool *vis) {
	bool anyVis = false;
	for (int l = 0; l < 4; l++) {
		bool front = true;
		if (depthRead) {
			if (e.clipSides && !e.clip[l]) {
				front = false;
			} else {
				float old = pick4(q.depth, e.slot[l]);
				front = affine ? (e.l0[l] < old) : (e.l0[l] > old);
			}
		}
		vis[l] = e.clip[l] && front;
		anyVis |= vis[l];
	}
	return anyVis;
}

// Shader of one quad of command c for all four lanes: RgbaMultiply's getPixels_2x2 with
// the vertex weights of the lanes (RgbaMultiply.h:74-175, shaderMethods.h:39-94).  The
// shader inputs were finished once per source triangle at setup.
__device__ __forceinline__ void shadeCommand(const FrameDev &f, int32_t c, const QuadEval &e, bool affine, uint32_t mask,
                                             float *r, float *g, float *b, float *a) {
	float wa[4], wb[4], wc[4];
	for (int l = 0; l < 4; l++) laneWeights(e, l, affine, wa[l], wb[l], wc[l]);
	const ShaderInputs si = f.shaders[c];
	shadeQuad(si, f.textures, wa, wb, wc, mask, r, g, b, a);
}

// The reference's shading of one quad (fillQuadSuper, fillerTemplates.h:154-187, with the
// RgbaMultiply shaders of RgbaMultiply.h:74-175).
__device__ void drawCommand(const FrameDev &f, const Command &cmd, int32_t c, const QuadEval &e,
                            QuadPixels<0> &q, bool colorWrite, bool depthRead, bool depthWrite, bool alphaFilter) {
	const bool affine = (cmd.flags & 1) != 0;
	bool vis[4];
	if (!quadVisibility<0>(e, q, depthRead, affine, vis)) return;
	if (colorWrite) {
		float r[4], g[4], b[4], a[4];
		const uint32_t mask = (vis[0] ? 1u : 0u) | (vis[1] ? 2u : 0u) | (vis[2] ? 4u : 0u) | (vis[3] ? 8u : 0u);
		shadeCommand(f, c, e, affine, mask, r, g, b, a);
		if (alphaFilter) {
			float tr[4], tg[4], tb[4], ta[4];
			for (int l = 0; l < 4; l++) {
				uint32_t old = (!e.clipSides || vis[l]) ? pick4(q.color, e.slot[l]) : 0u;
				unpackColor(old, tr[l], tg[l], tb[l], ta[l]);
			}
			for (int l = 0; l < 4; l++) {
				float opacity = a[l] * (1.0f / 255.0f);
				float inv = 1.0f - opacity;
				r[l] = (r[l] * opacity) + (tr[l] * inv);
				g[l] = (g[l] * opacity) + (tg[l] * inv);
				b[l] = (b[l] * opacity) + (tb[l] * inv);
				a[l] = (a[l] * opacity) + (ta[l] * inv);
			}
		}
		for (int l = 0; l < 4; l++) {
			if (vis[l]) {
				put4(q.color, e.slot[l], packSaturated(r[l], g[l], b[l], a[l]));
				q.colorDirty |= 1u << e.slot[l];
			}
		}
	}
	if (depthWrite) {
		for (int l = 0; l < 4; l++) {
			if (vis[l]) {
				put4(q.depth, e.slot[l], e.l0[l]);
				q.depthDirty |= 1u << e.slot[l];
			}
		}
	}
}

// ---------------------------------------------------------------------------------------
// Differentiable shading: colour = interpolated per-point RGB multipliers x bilinear sample
// of a float RGBA texture (level 0), alpha = the texture's alpha.  The texel choice and the
// 8-bit sub-texel weights are those of texture_sample_bilinear at the highest resolution
// (textureAPI.h:342-438); the adjoint below scatters through the same weights.
// ---------------------------------------------------------------------------------------

struct BilinearTaps {
	uint32_t index[4];  // texel indices: upper left, upper right, lower left, lower right
	float weight[4];
};

DH BilinearTaps bilinearTaps(int32_t log2w, int32_t log2h, float u, float v) {
	uint32_t scaleU = 256u << log2w, scaleV = 256u << log2h;
	uint32_t maskX = (1u << log2w) - 1u, maskY = (1u << log2h) - 1u;
	uint32_t subX = truncU32((u + 256.0f) * fromU32(scaleU)) - 128u;
	uint32_t subY = truncU32((v + 256.0f) * fromU32(scaleV)) - 128u;
	float fx = (float)(subX & 255u) * (1.0f / 256.0f), fy = (float)(subY & 255u) * (1.0f / 256.0f);
	uint32_t left = (subX >> 8) & maskX, top = (subY >> 8) & maskY;
	uint32_t right = (left + 1u) & maskX, bottom = (top + 1u) & maskY;
	BilinearTaps t;
	t.index[0] = (top << log2w) | left;
	t.index[1] = (top << log2w) | right;
	t.index[2] = (bottom << log2w) | left;
	t.index[3] = (bottom << log2w) | right;
	t.weight[0] = (1.0f - fx) * (1.0f - fy);
	t.weight[1] = fx * (1.0f - fy);
	t.weight[2] = (1.0f - fx) * fy;
	t.weight[3] = fx * fy;
	return t;
}

__device__ __forceinline__ float multiplier(const FrameDev &f, int32_t point, int ch) {
	return f.multipliers ? f.multipliers[point * 3 + ch] : 1.0f;
}

// records: the adjoint record of the quad's upper left pixel, with recordStride records per row (null
// when the frame keeps none).
__device__ void drawCommandDiff(const FrameDev &f, const Command &cmd, int32_t c, int32_t commandIndex, DiffRecord *records,
                                int32_t recordStride, const QuadEval &e, QuadPixels<1> &q, bool depthRead, bool depthWrite) {
	const bool affine = (cmd.flags & 1) != 0;
	bool vis[4];
	if (!quadVisibility<1>(e, q, depthRead, affine, vis)) return;
	const DiffInputs d = f.diffInputs[c];
	float m[3][3];
	for (int k = 0; k < 3; k++)
		for (int ch = 0; ch < 3; ch++) m[k][ch] = multiplier(f, d.point[k], ch);
	for (int l = 0; l < 4; l++) {
		if (!vis[l]) continue;
		float wa, wb, wc;
		laneWeights(e, l, affine, wa, wb, wc);
		float u = interp(d.u, wa, wb, wc), v = interp(d.v, wa, wb, wc);
		BilinearTaps taps = bilinearTaps(f.ftexLog2w, f.ftexLog2h, u, v);
		float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
		for (int k = 0; k < 4; k++) {
			const float4 texel = *(const float4 *)(f.ftexTexels + (size_t)taps.index[k] * 4);
			t[0] += taps.weight[k] * texel.x;
			t[1] += taps.weight[k] * texel.y;
			t[2] += taps.weight[k] * texel.z;
			t[3] += taps.weight[k] * texel.w;
		}
		const int s = e.slot[l];
		put4(q.r, s, (wa * m[0][0] + wb * m[1][0] + wc * m[2][0]) * t[0]);
		put4(q.g, s, (wa * m[0][1] + wb * m[1][1] + wc * m[2][1]) * t[1]);
		put4(q.b, s, (wa * m[0][2] + wb * m[1][2] + wc * m[2][2]) * t[2]);
		put4(q.a, s, t[3]);
		put4(q.vis, s, commandIndex * 4 + l);
		if (records) records[(s >> 1) * recordStride + (s & 1)] = DiffRecord{wb, wc, commandIndex * 4 + l, *f.forwardNumber};
		q.colorDirty |= 1u << s;
		if (depthWrite) {
			put4(q.depth, s, e.l0[l]);
			q.depthDirty |= 1u << s;
		}
	}
}

// The thread's index as a value the compiler cannot see through.  Taken at the top of a loop's
// body, the values derived from it there are computed in each trip instead of being held in
// registers across the loop (the visibility raster's per-chunk work would otherwise keep a
// dozen of them live through a whole tile, in scratch memory at five waves per SIMD).
__device__ __forceinline__ int32_t opaqueThreadIndex() {
	int32_t t = (int32_t)threadIdx.x;
	asm volatile("" : "+v"(t));
	return t;
}

constexpr int32_t ROUND_BINS_LOG2 = 8, ROUND_BINS = 1 << ROUND_BINS_LOG2;
// The largest index that ends the round after `last` (nextRound); -1 when no command is left.
template <int NT, int CAP>
__device__ __attribute__((noinline)) int32_t roundThreshold(const int32_t *src, int32_t n, int32_t last, int32_t *roundInfo, int32_t *hist) {
	static_assert(NT >= 64, "the first wavefront scans the bins");
	const int32_t t = (int32_t)threadIdx.x;
	if (t == 0) {
		roundInfo[0] = 0x7FFFFFFF;
		roundInfo[1] = -1;
		roundInfo[2] = 0;
	}
	__syncthreads();
	int32_t lowest = 0x7FFFFFFF, highest = -1;
	for (int32_t i = t; i < n; i += NT) {
		const int32_t v = src[i];
		if (v > last) lowest = tmin(lowest, v);
		highest = tmax(highest, v);
	}
	if (highest >= 0) {
		atomicMin(&roundInfo[0], lowest);
		atomicMax(&roundInfo[1], highest);
	}
	__syncthreads();
	int32_t lo = roundInfo[0], hi = roundInfo[1], threshold = -1;
	while (lo <= hi) {  // left with a threshold, or skipped when nothing remains
		const int32_t span = hi - lo, bits = span > 0 ? 32 - __builtin_clz((uint32_t)span) : 0;
		const int32_t shift = tmax(bits - ROUND_BINS_LOG2, 0);
		for (int32_t b = t; b < ROUND_BINS; b += NT) hist[b] = 0;
		__syncthreads();
		for (int32_t i = t; i < n; i += NT) {
			const int32_t v = src[i];
			if (v >= lo && v <= hi) atomicAdd(&hist[(v - lo) >> shift], 1);
		}
		__syncthreads();
		if (t < 64) {
			// Four bins per lane; counted: bins whose inclusive prefix stays within CAP.
			int32_t sum[4], total = 0;
#pragma unroll
			for (int k = 0; k < 4; k++) {
				total += hist[t * 4 + k];
				sum[k] = total;
			}
			int32_t before = total;
#pragma unroll
			for (int32_t offset = 1; offset < 64; offset <<= 1) {
				const int32_t y = __shfl_up(before, offset, 64);
				if (t >= offset) before += y;
			}
			before -= total;
			int32_t fit = 0, used = 0;
#pragma unroll
			for (int k = 0; k < 4; k++) {
				fit += __popcll(__ballot(before + sum[k] <= CAP));
				used += __popcll(__ballot(before + sum[k] == 0));
			}
			if (t == 0) {
				roundInfo[0] = fit;   // bins taken
				roundInfo[1] = used;  // empty bins before the first one in use
			}
		}
		__syncthreads();
		const int32_t fit = roundInfo[0], empty = roundInfo[1];
		__syncthreads();
		if (fit > empty) {
			threshold = (int32_t)tmin((uint32_t)hi, (uint32_t)lo + ((uint32_t)fit << shift) - 1u);
			break;
		}
		lo += empty << shift;  // the first bin in use
		hi = (int32_t)tmin((uint32_t)hi, (uint32_t)lo + (1u << shift) - 1u);
	}
	return threshold;
}

// Loads the next round of a tile's command list into LDS, sorted by command index: all of them when
// the list fits CAP, otherwise the commands in (last, threshold] for a threshold that keeps the round
// within CAP.  The threshold comes from a histogram of the remaining indices: the bins up to it hold
// at most CAP of them; when the first bin in use alone holds more, its range is cut into bins in turn
// (down to single indices, which are distinct).  A round reads the list three times (lowest and highest
// index, histogram, collection) and once more for each range cut again; searching the threshold by
// halving the index range read it 31 times, more than half the time of the tiles with over 256 commands (a list of 1 100: 676 of 1 122 us).  Every one of the workgroup's NT threads
// calls it; hist holds ROUND_BINS entries that are free here; returns the round's size.
template <int NT, int CAP = TILE_SORT_CAP>
__device__ int32_t nextRound(const int32_t *src, int32_t n, int32_t done, int32_t &last, int32_t *list, int32_t *roundInfo, int32_t *hist) {
	const int32_t t = threadIdx.x;
	int32_t take;
	if (done == 0 && n <= CAP) {
		for (int32_t i = t; i < n; i += NT) list[i] = src[i];
		take = n;
		last = 0x7FFFFFFE;
	} else {
		const int32_t threshold = roundThreshold<NT, CAP>(src, n, last, roundInfo, hist);
		for (int32_t i = t; i < n; i += NT) {
			const int32_t v = src[i];
			if (v > last && v <= threshold) list[atomicAdd(&roundInfo[2], 1)] = v;
		}
		__syncthreads();
		take = roundInfo[2];
		last = threshold;
	}
	__syncthreads();
	sortLds<NT>(list, take);
	return take;
}

// The three places where the in-order tile walk differs between the RGBA8 shaders (MODE 0)
// and the differentiable float shader (MODE 1), chosen by overload on the quad's pixel type.
__device__ __forceinline__ void loadQuadColor(QuadPixels<0> &q, int s, bool in, const CanvasDev &cv, const FrameDev &f, int32_t x, int32_t y) {
	q.color[s] = (in && cv.color && f.alphaAny) ? cv.color[(size_t)y * cv.colorStride + x] : 0u;
}
__device__ __forceinline__ void loadQuadColor(QuadPixels<1> &, int, bool, const CanvasDev &, const FrameDev &, int32_t, int32_t) {}

__device__ __forceinline__ void drawQuadCommand(const FrameDev &f, const Command &cmd, int32_t c, int32_t ci, const CanvasDev &cv,
                                                int32_t px, int32_t py, const QuadEval &e, QuadPixels<0> &q, bool colorWrite,
                                                bool depthRead, bool depthWrite, bool alphaFilter) {
	(void)ci;
	(void)cv;
	(void)px;
	(void)py;
	drawCommand(f, cmd, c, e, q, colorWrite, depthRead, depthWrite, alphaFilter);
}
__device__ __forceinline__ void drawQuadCommand(const FrameDev &f, const Command &cmd, int32_t c, int32_t ci, const CanvasDev &cv,
                                                int32_t px, int32_t py, const QuadEval &e, QuadPixels<1> &q, bool, bool depthRead,
                                                bool depthWrite, bool) {
	DiffRecord *records = f.diffRecords ? f.diffRecords + cv.recordBase + (int64_t)py * cv.width + px : nullptr;
	drawCommandDiff(f, cmd, c, c - f.canvasCommandBase[ci], records, cv.width, e, q, depthRead, depthWrite);
}

__device__ __forceinline__ void storeQuadColor(const QuadPixels<0> &q, int s, const CanvasDev &cv, int32_t x, int32_t y) {
	cv.color[(size_t)y * cv.colorStride + x] = q.color[s];
}
__device__ __forceinline__ void storeQuadColor(const QuadPixels<1> &q, int s, const CanvasDev &cv, int32_t x, int32_t y) {
	size_t p = (size_t)y * cv.diffStride + x;
	*(float4 *)(cv.diffColor + p * 4) = make_float4(q.r[s], q.g[s], q.b[s], q.a[s]);
	cv.visibility[p] = q.vis[s];
}

// One tile: load the lanes' pixels, draw every binned command in increasing command index
// (submission order), write back the pixels that changed.
template <int TW, int TH, int MODE>
__device__ void rasterTile(const FrameDev &f, int32_t tile, int32_t *list, RowInterval *rows, int32_t *roundInfo) {
	constexpr int32_t NL = (TW / 2) * (TH / 2);
	const int32_t n = f.tileCount[tile];
	const int32_t ci = findSegment(f.canvasTileEnd, f.canvasCount, tile);
	const CanvasDev cv = f.canvases[ci];
	const int32_t local = tile - cv.tileBase;
	const int32_t tileX0 = (local % cv.tilesX) * TW;
	const int32_t tileY0 = (local / cv.tilesX) * TH;
	const int32_t lane = threadIdx.x;
	const int32_t px = tileX0 + 2 * (lane % (TW / 2));
	const int32_t py = tileY0 + 2 * (lane / (TW / 2));
	const int32_t *src = tileListOf(f, tile);

	QuadPixels<MODE> q;
	q.colorDirty = q.depthDirty = 0;
	for (int s = 0; s < 4; s++) {
		int32_t x = px + (s & 1), y = py + (s >> 1);
		bool in = x < cv.width && y < cv.height;
		q.depth[s] = (in && cv.depth) ? cv.depth[(size_t)y * cv.depthStride + x] : 0.0f;
		loadQuadColor(q, s, in, cv, f, x, y);
	}

	int32_t last = -1;
	int32_t done = 0;
	while (done < n) {
		const int32_t take = nextRound<NL>(src, n, done, last, list, roundInfo, list + TILE_SORT_CAP);
		for (int32_t i = 0; i < take; i++) {
			const int32_t c = __builtin_amdgcn_readfirstlane(list[i]);
			const Command cmd = f.commands[c];
			const TaskDev &task = f.tasks[cmd.task];
			const bool solid = task.filter == 0;
			const bool colorWrite = MODE == 1 || cv.color != nullptr;
			const bool depthRead = cv.depth != nullptr;
			const bool depthWrite = cv.depth != nullptr && (solid || !colorWrite);
			const bool alphaFilter = colorWrite && !solid;
			// Rows of this command inside the tile: rasterizeTriangle over the aligned bound.
			const TriangleRows &tr = f.triangleRows[c];
			const int32_t alT = tr.alT, alB = tr.alB;
			__syncthreads();
			if (lane < TH) rows[lane] = triangleRow(tr, tileY0 + lane);
			__syncthreads();
			QuadEval e;
			if (py >= alT && py < alB && evalQuad(cmd, rows[py - tileY0], rows[py + 1 - tileY0], px, py, cv.height, e)) {
				drawQuadCommand(f, cmd, c, ci, cv, px, py, e, q, colorWrite, depthRead, depthWrite, alphaFilter);
			}
		}
		done += take;
		if (take == 0) break;
	}

	for (int s = 0; s < 4; s++) {
		int32_t x = px + (s & 1), y = py + (s >> 1);
		if (x >= cv.width || y >= cv.height) continue;
		if ((q.colorDirty >> s) & 1u) storeQuadColor(q, s, cv, x, y);
		if ((q.depthDirty >> s) & 1u) cv.depth[(size_t)y * cv.depthStride + x] = q.depth[s];
	}
}

// The raster kernel over the queue of non-empty tiles.  persistent = 0: workgroup b takes
// queue slot b (the grid covers every tile; surplus workgroups exit).  persistent = 1: a fixed
// grid whose workgroups pull slots from an atomic head until the queue is empty, so every
// workgroup reaches the exit once all tiles are handed out.
// The raster kernels start after every counter is final: workgroup 0 copies them to the
// frame's pinned host memory, which the host reads after the stream completes.
__device__ __forceinline__ void reportCounters(const FrameDev &f) {
	if (blockIdx.x == 0 && threadIdx.x < HOST_COUNTERS) f.hostCounters[threadIdx.x] = f.counters[threadIdx.x];
}

// A raster that leaves the next frame what k_frame_begin would (selfClean): the counters and the
// canvases' first-command indices come in two sets used by alternate frames, and workgroup 0
// resets the set this frame does not use; each tile's workgroup zeroes the tile's count once it
// has read it (tiles no workgroup visits have a count of zero).  The next frame then needs no
// begin kernel.  A frame whose raster returns early on an overflow leaves counts behind; the
// host runs the begin kernel after it.
__device__ __forceinline__ void resetNextCounters(const FrameDev &f) {
	if (!f.selfClean || blockIdx.x != 0) return;
	for (int32_t i = threadIdx.x; i < COUNTERS; i += blockDim.x) f.nextCounters[i] = 0;
	for (int32_t c = threadIdx.x; c < f.canvasCount; c += blockDim.x) f.nextCanvasBase[c] = 0x7FFFFFFF;
}

// Runs body(tile) over the tiles with commands -- every tile when the raster fills the
// canvases -- XCD by XCD.  The slots are the ordered queue of non-empty tiles after the scan,
// or the tiles themselves with direct bins (empty ones skipped).  Without persistence the grid
// has xcdGrid(tiles) workgroups and workgroup b takes the (b / 8)-th slot of XCD b % 8.
// Persistent workgroups pull slots from their own XCD's head and then from the other XCDs'
// heads; a head only grows and every XCD's slots end below the slot count, so all of them exit.
template <typename Body>
__device__ void forEachQueuedTile(const FrameDev &f, int32_t persistent, int32_t *slotLds, Body body) {
	const bool allTiles = f.clearInRaster || f.binCapacity > 0;
	const int32_t queued = allTiles ? f.tileTotal : f.counters[3];
	const int32_t x = (int32_t)(blockIdx.x % XCDS);
	if (!persistent) {
		const int32_t slot = xcdSlot(x, (int32_t)(blockIdx.x / XCDS));
		if (slot >= queued) return;
		const int32_t tile = allTiles ? slot : f.tileQueue[slot];
		if (f.clearInRaster || f.tileCount[tile] > 0) body(tile);
		return;
	}
	// First the tiles with long lists (phases 0 and 1): one of 1 100 commands takes about 500 us, the time
	// that the whole chip needs for 384 uneven jobs, and begun in tile order it ended 400 us after the
	// other tiles (raster 913 us; 842 now, as long as the longest list of 2 029 commands takes alone).
	// Then the others: persistent workgroups walk their own XCD's share first and help the other XCDs.
	for (int32_t phase = 0; phase < 2 + XCDS; phase++) {
		const bool longPhase = phase < 2;
		const int32_t xr = (x + phase - 2) % XCDS;
		const int32_t limit = longPhase ? f.counters[LONG_TILES + phase] : queued;
		int32_t *head = longPhase ? &f.counters[LONG_TILES + 2 + phase] : &f.counters[QUEUE_HEADS + QUEUE_HEAD_STRIDE * xr];
		while (limit > 0) {
			if (threadIdx.x == 0) {
				const int32_t ticket = atomicAdd(head, 1);
				*slotLds = longPhase ? ticket : xcdSlot(xr, ticket);
			}
			__syncthreads();
			const int32_t slot = *slotLds;
			__syncthreads();
			if (slot >= limit) break;
			const int32_t tile = longPhase ? f.longTiles[phase == 0 ? slot : f.tileTotal - 1 - slot] : (allTiles ? slot : f.tileQueue[slot]);
			const int32_t n = f.tileCount[tile];
			if (longPhase || (n <= LONG_LIST && (f.clearInRaster || n > 0))) body(tile);
			__syncthreads();
		}
	}
}

template <int TW, int TH>
__global__ void __launch_bounds__((TW / 2) * (TH / 2)) k_raster(FrameDev f, int32_t persistent) {
	if (f.mode == 1) return;  // the differentiable frames use k_raster_diff
	__shared__ int32_t list[TILE_SORT_CAP + ROUND_BINS];
	__shared__ RowInterval rows[TH];
	__shared__ int32_t roundInfo[3];
	__shared__ int32_t slotLds;
	reportCounters(f);
	if (f.counters[2]) return;  // an earlier stage ran out of room: leave the canvases untouched
	forEachQueuedTile(f, persistent, &slotLds, [&](int32_t tile) { rasterTile<TW, TH, 0>(f, tile, list, rows, roundInfo); });
}

template __global__ void k_raster<16, 16>(FrameDev, int32_t);
template __global__ void k_raster<32, 16>(FrameDev, int32_t);
template __global__ void k_raster<32, 32>(FrameDev, int32_t);

// ---------------------------------------------------------------------------------------
// Visibility raster for frames whose canvases hold commands of one projection each, perspective or
// orthogonal.
//
// Of Solid commands in the reference's order, a pixel ends with the colour and depth of the first
// reaching the best depth beyond the pixel's starting depth: a perspective command writes where
// its 1/W is strictly greater than the depth held at that moment, an orthogonal one where its W
// is strictly smaller (fillerTemplates.h:110-152), so the held depth is always the best value
// written so far and a later equal value loses.  That winner is found without walking the
// commands in order: every covered lane of every command offers the key (depth order << 32 |
// ~command) to the pixel with an LDS atomic max -- the order reversed on orthogonal canvases --
// and only the winning command is shaded for each pixel, with the same quad
// evaluation, weights and mip selection as the in-order walk.  Without a depth canvas the high
// half is the command's number, so the last covering command wins.  Commands run in chunks per tile;
// each chunk starts from the depths the previous one left.  Work is spread densely: one
// thread per (command, row) for the exact rows, per (command, covered quad) for the keys and
// per (command, covered quad) again for the shading of the lanes each command won.
//
// FORM_GENERAL: the frame has an orthogonal canvas or one of odd height.  An odd canvas's last row has
// no row below, and a quad's lower lanes there write the upper row's pixels after the upper lanes
// (fillerTemplates.h:287-323), so one command can leave a depth worse than its own other candidate and
// the argument above fails for that row alone.  The row's pixels (at most one row of the bottom tiles)
// are walked in submission order, a thread per quad; every other row goes through the keys.  Whole
// frames, while such frames were drawn in order and now: 1365x767 terrain 349 and 72 us, 1280x720
// orthogonal terrain 297 and 63 us.  Frames of even perspective canvases take kernels without that
// code, which made the persistent grid's 384-job batch 3 % slower.
//
// FORM_ALPHA: the frame has tasks with the Alpha filter, whose blending reads the colour held at that
// moment.  A chunk is then drawn in runs of one filter: runs of Solid commands through the keys, runs
// of Alpha commands by a walk in submission order with a thread per quad (blendRun).  It includes
// FORM_GENERAL.  One Alpha task is enough, and runs may be short: 1 000 objects of one triangle over a
// terrain at 1280x720, Solid and Alpha in turn, take the raster 51 us (135 in order), 10 objects of 100
// triangles 46 (147), and 64 jobs with one Alpha task among them 352 us (302 without it, 2 037 in order).
//
// Canvases that mix both projections (the depth test's direction changes between commands), canvases
// wider than 32767 pixels (rows are kept in 16 bits) and differentiable frames with the Alpha filter
// take the in-order kernel above.
// ---------------------------------------------------------------------------------------


// Keys order depths as floats compare: larger depth, larger key; -0 equals +0.
__device__ __forceinline__ uint32_t depthOrder(float d) {
	const uint32_t u = __float_as_uint(d + 0.0f);  // -0 + 0 = +0
	return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}

// A row interval in LDS: columns fit 16 bits (the visibility raster takes canvases up to
// 32767 pixels wide).
struct RowSpan { int16_t left, right; };
__device__ __forceinline__ RowSpan rowSpan(RowInterval r) { return RowSpan{(int16_t)r.left, (int16_t)r.right}; }
__device__ __forceinline__ RowInterval rowInterval(RowSpan r) { return RowInterval{r.left, r.right}; }

// CHUNK: commands staged and drawn at once.  Sixteen keep a 32x16 workgroup of the RGBA8 shaders
// within the LDS of eleven workgroups per CU.  The persistent
// grid's 32-pixel-wide tiles take 32 (at most eight workgroups per CU run anyway), and so do all
// tiles of the differentiable shader, whose scenes are denser, so that fewer tiles need a
// second chunk.
template <int TW, int TH, int P>
constexpr int32_t colorChunk() { return P != 0 && TW * TH >= 512 ? 32 : 16; }
constexpr int32_t DIFF_CHUNK = 32;

// Threads of a visibility-raster workgroup: four pixels of the tile per thread.  A 32x16 workgroup with
// chunks of 16 keeps to 14 080 bytes of LDS, so that eleven of them fit a CU.  The smaller limits that
// this takes cost nothing that shows, with 256 and 16 against 192 and 8: raster of a 1080p terrain with 8,
// 12 and 16 textures 52.9, 53.1 and 53.8 against 52.0, 52.7 and 53.4 us (16x16 tiles 56.9, 57.4 and 57.9
// against 53.4, 53.3 and 53.2); 256x256 canvases with tile lists of 60 to 130 commands on average,
// 141 to 282 against 139 to 281 us (16x16 tiles 157 to 320 against 158 to 325).
template <int TW, int TH, int CH> struct DeferShape {
	static constexpr int32_t NT = TW * TH / 4;
	static constexpr int32_t CHUNK = CH;                   // commands per chunk
	static constexpr bool TIGHT = TW * TH <= 512 && CH == 16;
	static constexpr int32_t LIST = TIGHT ? 192 : 256;     // commands sorted per round
	static constexpr int32_t TEXTURES = TIGHT ? 8 : 16;    // texture tables up to this size are read from LDS
};

static_assert(sizeof(TriangleRows) % 16 == 0 && sizeof(ShaderInputs) % 16 == 0 && sizeof(Command) % 16 == 0,
              "staged records are whole 16-byte units");

// The differentiable shader (drawCommandDiff) for the lanes in mask of one command's quad at
// (px, py), written straight to the float colour canvas with the visibility id base + lane.
__device__ void shadeDiffLanes(const FrameDev &f, const Command &ct, const DiffInputs &d, const QuadEval &e, uint32_t mask,
                               uint32_t slots, int32_t idBase, int32_t forward, const CanvasDev &cv, int32_t px, int32_t py) {
	const bool affine = (ct.flags & 1) != 0;
	float m[3][3];
	for (int c = 0; c < 3; c++)
		for (int ch = 0; ch < 3; ch++) m[c][ch] = multiplier(f, d.point[c], ch);
	for (int l = 0; l < 4; l++) {
		if (!((mask >> l) & 1u)) continue;
		const int32_t sl = (int32_t)((slots >> (2 * l)) & 3u);
		const int32_t x = px + (sl & 1), y = py + (sl >> 1);
		if (x >= cv.width || y >= cv.height) continue;
		float wa, wb, wc;
		laneWeights(e, l, affine, wa, wb, wc);
		const float u = interp(d.u, wa, wb, wc), v = interp(d.v, wa, wb, wc);
		const BilinearTaps taps = bilinearTaps(f.ftexLog2w, f.ftexLog2h, u, v);
		float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
		for (int k = 0; k < 4; k++) {
			const float4 texel = *(const float4 *)(f.ftexTexels + (size_t)taps.index[k] * 4);
			t[0] += taps.weight[k] * texel.x;
			t[1] += taps.weight[k] * texel.y;
			t[2] += taps.weight[k] * texel.z;
			t[3] += taps.weight[k] * texel.w;
		}
		const size_t p = (size_t)y * cv.diffStride + x;
		*(float4 *)(cv.diffColor + p * 4) = make_float4((wa * m[0][0] + wb * m[1][0] + wc * m[2][0]) * t[0],
		                                                (wa * m[0][1] + wb * m[1][1] + wc * m[2][1]) * t[1],
		                                                (wa * m[0][2] + wb * m[1][2] + wc * m[2][2]) * t[2], t[3]);
		cv.visibility[p] = idBase + l;
		if (f.diffRecords) f.diffRecords[cv.recordBase + (int64_t)y * cv.width + x] = DiffRecord{wb, wc, idBase + l, forward};
	}
}

// LDS of one visibility-raster workgroup.  The differentiable shader (MODE 1) writes its colours
// straight to the float canvas and reads no shader inputs or texture table, so it keeps none of
// them here, and more of its workgroups fit a CU.
template <int TW, int TH, int CH, int MODE> struct DeferLds {
	using S = DeferShape<TW, TH, CH>;
	static constexpr bool RGBA = MODE == 0;
	static constexpr int32_t PAIRS = S::CHUNK * (TH / 2);  // (command, row pair) slots of a chunk
	// Pass-1 items are found by table up to one per pixel per chunk (by binary search beyond).
	static constexpr int32_t ITEM_TABLE = TW * TH;
	using PairIndex = typename std::conditional<(PAIRS <= 256), uint8_t, uint16_t>::type;
	int32_t list[S::LIST];                       // the round's commands, sorted
	union {
		TriangleRows tr[S::CHUNK];               // the chunk's commands: row setup (until the rows are made),
		unsigned long long keys[TW * TH];        // then the pixels' (depth, command) keys
	};
	ShaderInputs si[RGBA ? S::CHUNK : 1];        // shader inputs,
	Command command[S::CHUNK];                  // weight planes and flags
	RowSpan rows[S::CHUNK * TH];                 // chunk command j, tile row r
	union {
		struct {                                 // during the rows:
			int32_t rowFirst[S::CHUNK];          // each command's first tile row inside its aligned bound
			int32_t rowStart[S::CHUNK + 1];      // exclusive prefix of those rows per command
		};
		struct {                                 // from the pairs to pass 2:
			uint8_t pairStart[PAIRS];            // first quad column of each pair, from the tile's left
			int16_t pairOffset[PAIRS + 1];       // exclusive prefix of quads per pair
			PairIndex pairOfItem[ITEM_TABLE];    // the pair of each of the first ITEM_TABLE pass-1 items
		};
	};
	float depth[TW * TH];                        // the tile's depths as they stand
	uint32_t color[RGBA ? TW * TH : 1];          // the drawn pixels' colours
	uint32_t dirty[TW * TH / 32];                // pixels written, one bit each
	uint32_t chunkWon[RGBA ? TW * TH / 32 : 1];  // pixels the current chunk's commands won
	int32_t scan[S::NT / 64];                    // wavefront totals of the prefix sums
	TextureDesc textures[RGBA ? S::TEXTURES : 1];
	int32_t roundInfo[4];
	int32_t slot;
};

// Copies element list[c0 + j] of a global array of T into dst[j], for every chunk command j, with loads
// that write LDS directly (no registers hold the data), 16 bytes per lane.  Each wave instruction fills
// 64 consecutive units of dst.  The caller waits for them (stageWait) before reading dst.
template <int NT, typename T>
__device__ __forceinline__ void stageToLds(T *dst, const uint8_t *src, const int32_t *list, int32_t c0, int32_t cn) {
	constexpr int32_t UNITS = (int32_t)(sizeof(T) / 16);
	const int32_t total = cn * UNITS;
	const int32_t lane = (int32_t)(threadIdx.x & 63);
	for (int32_t base = (int32_t)(threadIdx.x & ~63u); base < total; base += NT) {
		const int32_t q = base + lane;
		if (q < total) {
			const int32_t j = q / UNITS, u = q % UNITS;
			const uint8_t *g = src + (size_t)list[c0 + j] * sizeof(T) + u * 16;
			__builtin_amdgcn_global_load_lds((const void *)g, (void *)((uint8_t *)dst + (size_t)base * 16), 16, 0, 0);
		}
	}
}

// Waits for this thread's LDS-direct loads; a barrier then publishes them to the workgroup.
__device__ __forceinline__ void stageWait() { __builtin_amdgcn_s_waitcnt(0); }


// A canvas store: the pointer, read from memory, is known to be global.
template <typename T> __device__ __forceinline__ void storeGlobal(T *p, T value) { *(__attribute__((address_space(1))) T *)p = value; }

// The low half of a key of chunk command j, below which the canvas's own value (all ones) ranks first
// and equal depths go to the earlier command.  Without a depth canvas the high half is j + 1.
__device__ __forceinline__ uint32_t keyOfCommand(int32_t j) { return 0xFFFFFFFEu - (uint32_t)j; }

// Index of the segment holding item it in an exclusive prefix of count + 1 entries.
template <typename T>
__device__ __forceinline__ int32_t segmentOf(const T *offset, int32_t count, int32_t it) {
	int32_t lo = 0, hi = count - 1;
	while (lo < hi) {
		const int32_t mid = (lo + hi + 1) >> 1;
		if (offset[mid] <= it) lo = mid; else hi = mid - 1;
	}
	return lo;
}

// The lanes of command j's quad, whose upper left pixel has its key at key[0], that won their pixels.
// A lane's pixel is the lane's own except in an odd canvas's last row (oddRow), where the key's high
// half says which of a column's two lanes wrote it.
template <int TW, bool GENERAL>
__device__ __forceinline__ uint32_t lanesWon(const unsigned long long *key, int32_t j, bool oddRow) {
	const uint32_t *half = (const uint32_t *)key;
	const uint32_t own = keyOfCommand(j);
	if (GENERAL && oddRow)
		return (half[0] == own ? 1u << (2 * (half[1] & 1u)) : 0u) | (half[2] == own ? 2u << (2 * (half[3] & 1u)) : 0u);
	return (half[0] == own ? 1u : 0u) | (half[2] == own ? 2u : 0u) | (half[2 * TW] == own ? 4u : 0u) | (half[2 * TW + 2] == own ? 8u : 0u);
}

// The Alpha filter's commands [j0, j1) of a chunk over the tile's colours and depths in LDS: a thread
// per quad walks them in submission order (drawCommand's tests, shading and blending), no thread needs
// another's pixels, and the commands' rows and inputs are staged, so nothing separates two commands.
// The in-order raster, which this replaces, made each command's rows between two barriers of its own.
template <int TW, int TH, typename Lds>
__device__ __forceinline__ void blendRun(Lds &s, int32_t j0, int32_t j1, int32_t tileX0, int32_t tileY0, const CanvasDev &cv,
                                         const TextureTable &textures, bool depthRead) {
	const int32_t t = opaqueThreadIndex();
	const int32_t qx = 2 * (t % (TW / 2)), qy = 2 * (t / (TW / 2)), first = qy * TW + qx;
	uint32_t drawn = 0;
	for (int32_t j = j0; j < j1; j++) {
		QuadEval e;
		if (!evalQuad(s.command[j].plane, rowInterval(s.rows[j * TH + qy]), rowInterval(s.rows[j * TH + qy + 1]), tileX0 + qx, tileY0 + qy,
		              cv.height, e))
			continue;
		const bool affine = (s.command[j].flags & 1) != 0;
		uint32_t visible = 0, old[4];
#pragma unroll
		for (int l = 0; l < 4; l++) {
			const int32_t p = first + (e.slot[l] >> 1) * TW + (e.slot[l] & 1);
			bool front = true;
			if (depthRead) {
				const float held = s.depth[p];
				front = affine ? e.l0[l] < held : e.l0[l] > held;
			}
			if (e.clip[l] && front) visible |= 1u << l;
			old[l] = s.color[p];
		}
		if (!visible) continue;
		float wa[4], wb[4], wc[4];
		for (int l = 0; l < 4; l++) laneWeights(e, l, affine, wa[l], wb[l], wc[l]);
		const uint32_t mip = quadMip(s.si[j], textures, wa, wb, wc);
#pragma unroll
		for (int l = 0; l < 4; l++) {
			if (!((visible >> l) & 1u)) continue;
			float r, g, b, a, tr, tg, tb, ta;
			shadeChannels(s.si[j], textures, wa[l], wb[l], wc[l], mip, r, g, b, a);
			unpackColor(old[l], tr, tg, tb, ta);
			const float opacity = a * (1.0f / 255.0f), inv = 1.0f - opacity;
			r = (r * opacity) + (tr * inv);
			g = (g * opacity) + (tg * inv);
			b = (b * opacity) + (tb * inv);
			a = (a * opacity) + (ta * inv);
			s.color[first + (e.slot[l] >> 1) * TW + (e.slot[l] & 1)] = packSaturated(r, g, b, a);
			drawn |= 1u << e.slot[l];
		}
	}
	if (drawn) {
		atomicOr(&s.dirty[first >> 5], (drawn & 3u) << (first & 31));
		atomicOr(&s.dirty[(first + TW) >> 5], (drawn >> 2) << ((first + TW) & 31));
	}
}

// MODE 0: the RGBA8 shaders into the colour canvas.  MODE 1: the differentiable float shader
// into the float colour canvas plus the visibility id of each pixel's winning lane.
template <int TW, int TH, int MODE, int FORM, int CH>
__device__ void rasterTileDeferred(const FrameDev &f, int32_t tile, DeferLds<TW, TH, CH, MODE> &s, const TextureTable &textures) {
	using S = DeferShape<TW, TH, CH>;
	constexpr bool GENERAL = FORM != FORM_PLAIN, ALPHA = FORM == FORM_ALPHA;
	constexpr int32_t NT = S::NT, CHUNK = S::CHUNK;
	constexpr int32_t NP = TW * TH, RP = TH / 2;
	constexpr int32_t PAIRS = DeferLds<TW, TH, CH, MODE>::PAIRS;
	constexpr int32_t ITEM_TABLE = DeferLds<TW, TH, CH, MODE>::ITEM_TABLE;
	constexpr int32_t PAIRS_PER_THREAD = PAIRS / NT > 0 ? PAIRS / NT : 1;
	const int32_t n = f.tileCount[tile];
	const int32_t ci = findSegment(f.canvasTileEnd, f.canvasCount, tile);
	const CanvasDev cv = f.canvases[ci];
	const int32_t local = tile - cv.tileBase;
	const int32_t tileX0 = (local % cv.tilesX) * TW;
	const int32_t tileY0 = (local / cv.tilesX) * TH;
	const int32_t t = threadIdx.x;
	const int32_t *src = tileListOf(f, tile);
	const bool colorWrite = MODE == 0 && cv.color != nullptr;
	const bool depthRead = cv.depth != nullptr;
	const uint32_t flip = GENERAL && cv.affine ? ~0u : 0u;  // orthogonal canvases: the smaller depth wins
	const int32_t forward = MODE == 1 && f.diffRecords ? *f.forwardNumber : 0;

	for (int32_t p = t; p < NP; p += NT) {
		if (f.clearInRaster) {
			s.depth[p] = f.clearDepth;
		} else {
			const int32_t x = tileX0 + p % TW, y = tileY0 + p / TW;
			s.depth[p] = (depthRead && x < cv.width && y < cv.height) ? cv.depth[(size_t)y * cv.depthStride + x] : 0.0f;
		}
		if (ALPHA && colorWrite) {  // blending reads the colours that are there
			const int32_t x = tileX0 + p % TW, y = tileY0 + p / TW;
			s.color[p] = f.clearInRaster ? f.clearColor : (x < cv.width && y < cv.height ? cv.color[(size_t)y * cv.colorStride + x] : 0u);
		}
	}
	// With the fill fused in, the pixels that no command draws take the fill values at the write-back.
	for (int32_t w = t; w < NP / 32; w += NT) s.dirty[w] = 0u;
	if (n == 0) __syncthreads();  // an empty tile only takes the fill: no round's barrier comes before the write-back

	int32_t last = -1;
	int32_t done = 0;
	while (done < n) {
		const int32_t take = nextRound<NT, S::LIST>(src, n, done, last, s.list, s.roundInfo, (int32_t *)s.keys);
		for (int32_t c0 = 0; c0 < take; c0 += CHUNK) {
			const int32_t t = opaqueThreadIndex();
			const int32_t cn = take - c0 < CHUNK ? take - c0 : CHUNK;
			// The chunk's row setups, shader inputs and weight planes into LDS.
			stageToLds<NT>(s.tr, (const uint8_t *)f.triangleRows, s.list, c0, cn);
			if (colorWrite) stageToLds<NT>(s.si, (const uint8_t *)f.shaders, s.list, c0, cn);
			stageToLds<NT>(s.command, (const uint8_t *)f.commands, s.list, c0, cn);
			stageWait();
			__syncthreads();
			// Rows of every chunk command in the tile: empty outside the command's aligned bound,
			// and inside it the exact interval of rasterizeTriangle, one (command, row) per thread.
			for (int32_t idx = t; idx < cn * TH; idx += NT) s.rows[idx] = RowSpan{0, 0};
			if (t < 64) {
				int32_t first = 0, count = 0;
				if (t < cn) {
					first = tmin(tmax(s.tr[t].alT - tileY0, 0), TH);
					count = tmax(tmin(tmax(s.tr[t].alB - tileY0, 0), TH) - first, 0);
				}
				int32_t x = count;
#pragma unroll
				for (int32_t offset = 1; offset < 64; offset <<= 1) {
					const int32_t y = __shfl_up(x, offset, 64);
					if (t >= offset) x += y;
				}
				if (t < cn) {
					s.rowFirst[t] = first;
					s.rowStart[t] = x - count;
				}
				if (t == cn - 1) s.rowStart[cn] = x;
			}
			__syncthreads();
			const int32_t rowItems = s.rowStart[cn];
			for (int32_t it = t; it < rowItems; it += NT) {
				const int32_t j = segmentOf(s.rowStart, cn, it);
				const int32_t r = s.rowFirst[j] + (it - s.rowStart[j]);
				s.rows[j * TH + r] = rowSpan(triangleRow(s.tr[j], tileY0 + r));
			}
			__syncthreads();
			// Runs of commands of one filter, in submission order (one run for all without the Alpha filter).
			for (int32_t j0 = 0, j1 = cn; j0 < cn; j0 = j1) {
				if (ALPHA && colorWrite) {
					const int32_t lane = t & 63;
					const uint64_t blended = __ballot(lane < cn && (s.command[lane < cn ? lane : 0].flags & 2) != 0);
					const bool blends = ((blended >> j0) & 1u) != 0;
					const uint64_t other = (blends ? ~blended : blended) >> j0;
					j1 = other != 0 ? tmin(j0 + (int32_t)__builtin_ctzll(other), cn) : cn;
					if (blends) {
						blendRun<TW, TH>(s, j0, j1, tileX0, tileY0, cv, textures, depthRead);
						__syncthreads();
						continue;
					}
				}
				// Keys start at the held depth with the lowest command part above every command's,
				// so only a strictly greater depth replaces it; a NaN depth is never replaced.
				for (int32_t p = t; p < NP; p += NT) {
					const float d = s.depth[p];
					s.keys[p] = !depthRead ? 0ull : (d != d ? ~0ull : (((unsigned long long)(depthOrder(d) ^ flip) << 32) | 0xFFFFFFFFull));
				}
				if (MODE == 0)
					for (int32_t w = t; w < NP / 32; w += NT) s.chunkWon[w] = 0u;
				// Quads of each (command, row pair) inside the tile: the outer span of the row pair
				// (fillShapeSuper), cut to the tile's columns.
				int32_t pairCount[PAIRS_PER_THREAD];
				int32_t threadSum = 0;
				for (int32_t k = 0; k < PAIRS_PER_THREAD; k++) {
					const int32_t pr = t * PAIRS_PER_THREAD + k;
					const int32_t j = pr / RP, rp = pr % RP;
					int32_t count = 0, x0 = 0;
					if (pr < PAIRS && j < j1 && (!ALPHA || j >= j0)) {
						const RowInterval upper = rowInterval(s.rows[j * TH + 2 * rp]), lower = rowInterval(s.rows[j * TH + 2 * rp + 1]);
						if (upper.right > upper.left || lower.right > lower.left) {
							const int32_t outerBlockStart = (int32_t)((uint32_t)tmin(upper.left, lower.left) & ~1u);
							const int32_t outerBlockEnd = (int32_t)(((uint32_t)tmax(upper.right, lower.right) + 1u) & ~1u);
							x0 = tmax(outerBlockStart, tileX0);
							const int32_t x1 = tmin(outerBlockEnd, tileX0 + TW);
							count = x1 > x0 ? (x1 - x0) >> 1 : 0;
						}
					}
					if (pr < PAIRS) s.pairStart[pr] = (uint8_t)(x0 - tileX0);
					pairCount[k] = count;
					threadSum += count;
				}
				int32_t before;
				const int32_t items = workgroupPrefix<NT>(threadSum, before, s.scan);
				for (int32_t k = 0; k < PAIRS_PER_THREAD; k++) {
					const int32_t pr = t * PAIRS_PER_THREAD + k;
					if (pr < PAIRS) s.pairOffset[pr] = (int16_t)before;
					for (int32_t i = before; i < before + pairCount[k] && i < ITEM_TABLE; i++)
						s.pairOfItem[i] = (typename DeferLds<TW, TH, CH, MODE>::PairIndex)pr;
					before += pairCount[k];
				}
				if (t == 0) s.pairOffset[PAIRS] = (int16_t)items;
				__syncthreads();
				// Pass 1: one (command, quad) item per thread offers the covered lanes' keys.
				for (int32_t it = t; it < items; it += NT) {
					const int32_t pr = it < ITEM_TABLE ? (int32_t)s.pairOfItem[it] : segmentOf(s.pairOffset, PAIRS, it);
					const int32_t j = pr / RP, rp = pr % RP;
					const int32_t px = tileX0 + s.pairStart[pr] + 2 * (it - s.pairOffset[pr]);
					const int32_t py = tileY0 + 2 * rp;
					if (GENERAL && py + 1 >= cv.height) continue;  // walked below
					QuadEval e;
					const bool ok = evalQuad(s.command[j].plane, rowInterval(s.rows[j * TH + 2 * rp]), rowInterval(s.rows[j * TH + 2 * rp + 1]),
					                         px, py, cv.height, e);
					if (!ok) continue;
					// A lane whose row misses the quad is clipped, so a lane that counts is its own pixel.
					unsigned long long *key = &s.keys[2 * rp * TW + px - tileX0];
	#pragma unroll
					for (int l = 0; l < 4; l++) {
						const float d = e.l0[l];
						const bool offers = (!e.clipSides || e.clip[l]) && (!depthRead || d == d);
						const uint32_t rank = depthRead ? depthOrder(d) ^ flip : (uint32_t)(j + 1);
						if (offers) atomicMax(&key[(l >> 1) * TW + (l & 1)], ((unsigned long long)rank << 32) | keyOfCommand(j));
					}
				}
				// The odd canvas's last row: both lanes of a column test the depth held before the
				// command, then the upper one writes, then the lower one (drawCommand).  The key keeps
				// the last command that wrote and, in the high half, which of the two lanes it was.
				if (GENERAL && (cv.height & 1) && tileY0 + TH > cv.height && t < TW / 2) {
					const int32_t py = cv.height - 1, px = tileX0 + 2 * t;
					float held[2] = {s.depth[(py - tileY0) * TW + 2 * t], s.depth[(py - tileY0) * TW + 2 * t + 1]};
					int32_t winner[2] = {-1, -1}, lower[2] = {0, 0};
					for (int32_t j = j0; j < j1; j++) {
						const RowSpan upperRow = s.rows[j * TH + py - tileY0];
						if (upperRow.right <= upperRow.left) continue;
						QuadEval e;
						if (!evalQuad(s.command[j].plane, rowInterval(upperRow), rowInterval(s.rows[j * TH + py - tileY0 + 1]), px, py, cv.height, e)) continue;
	#pragma unroll
						for (int i = 0; i < 2; i++) {
							const float old = held[i];
	#pragma unroll
							for (int half = 0; half < 2; half++) {
								const int l = 2 * half + i;
								if (!e.clip[l]) continue;
								if (depthRead && !(cv.affine ? e.l0[l] < old : e.l0[l] > old)) continue;
								held[i] = e.l0[l];
								winner[i] = j;
								lower[i] = half;
							}
						}
					}
	#pragma unroll
					for (int i = 0; i < 2; i++)
						if (winner[i] >= 0)
							s.keys[(py - tileY0) * TW + 2 * t + i] = ((unsigned long long)lower[i] << 32) | keyOfCommand(winner[i]);
				}
				__syncthreads();
				if (MODE == 0) {
					// Pass 2: each item that won a lane evaluates its quad again (keeping pass 1's
					// evaluations would cost more registers than the evaluation), writes the won lanes'
					// depths, and leaves for every won pixel its weights (in the pixel's key) and its command
					// and the quad's mip level (in its colour, about to be replaced), so that pass 3 shades
					// each pixel once with all threads busy.  Only a pixel's winner replaces its key, and the
					// weight that takes the low half's place is no other command's: those halves are NaNs that
					// no arithmetic gives, and a NaN weight is stored as the usual one.  So no barrier
					// separates the reading of the keys from their replacement.
					for (int32_t it = t; it < items; it += NT) {
						const int32_t pr = it < ITEM_TABLE ? (int32_t)s.pairOfItem[it] : segmentOf(s.pairOffset, PAIRS, it);
						const int32_t j = pr / RP, rp = pr % RP;
						const int32_t qx = s.pairStart[pr] + 2 * (it - s.pairOffset[pr]), qy = 2 * rp;
						const int32_t first = qy * TW + qx;
						const bool oddRow = GENERAL && tileY0 + qy + 1 >= cv.height;
						const uint32_t mask = lanesWon<TW, GENERAL>(&s.keys[first], j, oddRow);
						if (!mask) continue;
						QuadEval e;
						if (!evalQuad(s.command[j].plane, rowInterval(s.rows[j * TH + qy]), rowInterval(s.rows[j * TH + qy + 1]), tileX0 + qx,
						              tileY0 + qy, cv.height, e))
							continue;
						// The won pixels of the quad's two rows, as bits of their words.
						const uint32_t upper = (oddRow ? mask | (mask >> 2) : mask) & 3u, lower = oddRow ? 0u : mask >> 2;
						atomicOr(&s.chunkWon[first >> 5], upper << (first & 31));
						atomicOr(&s.chunkWon[(first + TW) >> 5], lower << ((first + TW) & 31));
	#pragma unroll
						for (int l = 0; l < 4; l++)
							if ((mask >> l) & 1u) s.depth[first + (oddRow ? 0 : (l >> 1) * TW) + (l & 1)] = e.l0[l];
						if (colorWrite) {
							const bool affine = (s.command[j].flags & 1) != 0;
							float wa[4], wb[4], wc[4];
							for (int l = 0; l < 4; l++) laneWeights(e, l, affine, wa[l], wb[l], wc[l]);
							const uint32_t shade = (uint32_t)j | (quadMip(s.si[j], textures, wa, wb, wc) << 5);
	#pragma unroll
							for (int l = 0; l < 4; l++) {
								if (!((mask >> l) & 1u)) continue;
								const int32_t p = first + (oddRow ? 0 : (l >> 1) * TW) + (l & 1);
								const uint32_t weight = wb[l] == wb[l] ? __float_as_uint(wb[l]) : 0x7FC00000u;
								s.keys[p] = ((unsigned long long)__float_as_uint(wc[l]) << 32) | weight;
								s.color[p] = shade;
							}
						}
					}
					__syncthreads();
					// Pass 3: every pixel won in this chunk, shaded once.
					for (int32_t w = t; w < NP / 32; w += NT) s.dirty[w] |= s.chunkWon[w];
					if (colorWrite) {
						for (int32_t p = t; p < NP; p += NT) {
							if (!((s.chunkWon[p >> 5] >> (p & 31)) & 1u)) continue;
							const uint32_t shade = s.color[p];
							const unsigned long long weights = s.keys[p];
							const float wb = __uint_as_float((uint32_t)weights), wc = __uint_as_float((uint32_t)(weights >> 32));
							s.color[p] = shadePixel(s.si[shade & 31u], textures, 1.0f - (wb + wc), wb, wc, shade >> 5);
						}
					}
				} else {
					// Pass 2 of the differentiable shader: the same items, evaluated again; each writes
					// the lanes whose pixels its command won, with the quad's weights as in the in-order
					// walk.  A pixel has one winner, so exactly one item writes it.
					for (int32_t it = t; it < items; it += NT) {
						const int32_t pr = it < ITEM_TABLE ? (int32_t)s.pairOfItem[it] : segmentOf(s.pairOffset, PAIRS, it);
						const int32_t j = pr / RP, rp = pr % RP;
						const int32_t qx = s.pairStart[pr] + 2 * (it - s.pairOffset[pr]), qy = 2 * rp;
						const uint32_t mask = lanesWon<TW, GENERAL>(&s.keys[qy * TW + qx], j, GENERAL && tileY0 + qy + 1 >= cv.height);
						if (!mask) continue;
						QuadEval e;
						if (!evalQuad(s.command[j].plane, rowInterval(s.rows[j * TH + qy]), rowInterval(s.rows[j * TH + qy + 1]), tileX0 + qx,
						              tileY0 + qy, cv.height, e))
							continue;
						// Depths first, so that only the weights and the won lanes' pixels outlive the quad
						// evaluation while the colours are made.
						uint32_t slots = 0;
						for (int l = 0; l < 4; l++) {
							if (!((mask >> l) & 1u)) continue;
							const int32_t sl = e.slot[l];
							const int32_t p = (qy + (sl >> 1)) * TW + qx + (sl & 1);
							s.depth[p] = e.l0[l];
							atomicOr(&s.dirty[p >> 5], 1u << (p & 31));
							slots |= (uint32_t)sl << (2 * l);
						}
						const int32_t id = (s.list[c0 + j] - f.canvasCommandBase[ci]) * 4;
						shadeDiffLanes(f, s.command[j], f.diffInputs[s.list[c0 + j]], e, mask, slots, id, forward, cv, tileX0 + qx, tileY0 + qy);
					}
				}
				__syncthreads();
			}
		}
		done += take;
		if (take == 0) break;
	}

	for (int32_t p = t; p < NP; p += NT) {
		const bool drawn = ((s.dirty[p >> 5] >> (p & 31)) & 1u) != 0;
		if (!drawn && !f.clearInRaster) continue;
		const int32_t x = tileX0 + p % TW, y = tileY0 + p / TW;
		if (x >= cv.width || y >= cv.height) continue;
		if (colorWrite) storeGlobal(cv.color + (size_t)y * cv.colorStride + x, drawn ? s.color[p] : f.clearColor);
		if (depthRead) storeGlobal(cv.depth + (size_t)y * cv.depthStride + x, s.depth[p]);
		if (MODE == 1 && !drawn) {  // the fill values of k_clear_canvases
			const size_t q = (size_t)y * cv.diffStride + x;
			*(float4 *)(cv.diffColor + q * 4) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
			cv.visibility[q] = -1;
		}
	}
	if (f.selfClean && t == 0) f.tileCount[tile] = 0;  // read by this workgroup alone, long before
}

// Waves per SIMD: as many as the LDS leaves room for, since the raster waits for memory and barriers as
// much as for its own instructions (4K terrain 138 us with ten 32x16 workgroups per CU, 133 with eleven).
// P = 1: persistent workgroups, at four waves per SIMD (a persistent grid holds at most eight workgroups
// per CU).  The two forms are separate kernels so
// that each gets its own register allocation (the persistent loop keeps more values live).
// The Alpha form's walk keeps a quad and four colours in registers.
template <int TW, int TH, int P, int FORM>
constexpr int32_t rasterWaves() { return P || FORM == FORM_ALPHA ? 4 : (TW * TH == 512 ? 6 : 5); }
template <int TW, int TH, int P, int FORM>
__global__ void __launch_bounds__(TW * TH / 4) __attribute__((amdgpu_waves_per_eu(rasterWaves<TW, TH, P, FORM>(), rasterWaves<TW, TH, P, FORM>()))) k_raster_deferred(FrameDev f) {
	__shared__ DeferLds<TW, TH, colorChunk<TW, TH, P>(), 0> s;
	reportCounters(f);
	resetNextCounters(f);
	if (f.counters[2]) return;  // an earlier stage ran out of room: leave the canvases untouched
	// Small texture tables are read from LDS by the shading.
	const bool ldsTextures = f.textureCount <= DeferShape<TW, TH, colorChunk<TW, TH, P>()>::TEXTURES;
	if (ldsTextures) {
		constexpr int32_t W = (int32_t)(sizeof(TextureDesc) / 4);
		for (int32_t i = threadIdx.x; i < f.textureCount * W; i += TW * TH / 4)
			((uint32_t *)s.textures)[i] = ((const uint32_t *)f.textures)[i];
		__syncthreads();
	}
	const TextureTable textures = {(const __attribute__((address_space(3))) TextureDesc *)s.textures,
	                               (const __attribute__((address_space(1))) TextureDesc *)f.textures, ldsTextures};
	forEachQueuedTile(f, P, &s.slot, [&](int32_t tile) { rasterTileDeferred<TW, TH, 0, FORM>(f, tile, s, textures); });
}

// Waves per SIMD of the differentiable visibility raster: six for 32x16 tiles of one workgroup
// each (16 B of scratch; 8-view fit forward raster 169 us with five, 160 with six), four for the others,
// where more costs more in scratch than it gains.
template <int TW, int TH, int P>
constexpr int32_t diffWaves() { return P == 0 && TW * TH == 512 ? 6 : 4; }

// The differentiable forward by the visibility raster.
template <int TW, int TH, int P, int FORM>
__global__ void __launch_bounds__(TW * TH / 4) __attribute__((amdgpu_waves_per_eu(diffWaves<TW, TH, P>(), diffWaves<TW, TH, P>()))) k_raster_deferred_diff(FrameDev f) {
	__shared__ DeferLds<TW, TH, DIFF_CHUNK, 1> s;
	reportCounters(f);
	if (f.counters[2]) return;
	forEachQueuedTile(f, P, &s.slot, [&](int32_t tile) { rasterTileDeferred<TW, TH, 1, FORM>(f, tile, s, TextureTable()); });
}

#define DEFERRED_SHAPE(TW, TH, FORM)                                    \
	template __global__ void k_raster_deferred<TW, TH, 0, FORM>(FrameDev); \
	template __global__ void k_raster_deferred<TW, TH, 1, FORM>(FrameDev);
#define DEFERRED_DIFF_SHAPE(TW, TH, FORM)                                    \
	template __global__ void k_raster_deferred_diff<TW, TH, 0, FORM>(FrameDev); \
	template __global__ void k_raster_deferred_diff<TW, TH, 1, FORM>(FrameDev);
#define EVERY_TILE_SHAPE(KIND, FORM) KIND(16, 16, FORM) KIND(32, 16, FORM) KIND(32, 32, FORM)
EVERY_TILE_SHAPE(DEFERRED_SHAPE, FORM_PLAIN)
EVERY_TILE_SHAPE(DEFERRED_SHAPE, FORM_GENERAL)
EVERY_TILE_SHAPE(DEFERRED_SHAPE, FORM_ALPHA)
EVERY_TILE_SHAPE(DEFERRED_DIFF_SHAPE, FORM_PLAIN)
EVERY_TILE_SHAPE(DEFERRED_DIFF_SHAPE, FORM_GENERAL)
#undef EVERY_TILE_SHAPE
#undef DEFERRED_DIFF_SHAPE
#undef DEFERRED_SHAPE

// The differentiable forward: the same tile walk with the float shader, persistent or not.
template <int TW, int TH>
__global__ void __launch_bounds__((TW / 2) * (TH / 2)) k_raster_diff(FrameDev f, int32_t persistent) {
	__shared__ int32_t list[TILE_SORT_CAP + ROUND_BINS];
	__shared__ RowInterval rows[TH];
	__shared__ int32_t roundInfo[3];
	__shared__ int32_t slotLds;
	reportCounters(f);
	if (f.counters[2]) return;
	forEachQueuedTile(f, persistent, &slotLds, [&](int32_t tile) { rasterTile<TW, TH, 1>(f, tile, list, rows, roundInfo); });
}

template __global__ void k_raster_diff<16, 16>(FrameDev, int32_t);
template __global__ void k_raster_diff<32, 16>(FrameDev, int32_t);
template __global__ void k_raster_diff<32, 32>(FrameDev, int32_t);

// ---------------------------------------------------------------------------------------
// Depth-only tiles (model_renderDepth: executeTriangleDrawingDepth, renderCore.cpp:344-387).
//
// Each row of a draw command starts at the depth of its first pixel from the weight plane and
// adds the plane's x step once per pixel; a pixel takes the value when it is strictly greater
// than the depth held (perspective, 1/W) or strictly smaller (orthogonal, W).  The tile's
// depths live in LDS as 64-bit keys: the depth's order in the high half (reversed for
// orthogonal cameras, +0 and -0 equal), and below it the command's priority -- the held value
// first, then the tile's commands in submission order -- and the sign of a zero depth.  An
// atomic max over the keys of every covered pixel of every command leaves, per pixel, the
// first command to reach the best depth: the value the in-order walk keeps, including which of
// +0 and -0 when they tie.  NaN is never written and a held NaN is never replaced.  One thread
// per (command, row): the row is exact (rasterizeTriangle), and its depth chain runs from the
// row's first pixel, so columns left of the tile are stepped over without being written.
// ---------------------------------------------------------------------------------------
constexpr uint32_t DEPTH_HELD_PRIORITY = 0x7FFFFFFFu;

__device__ __forceinline__ uint32_t depthOnlyOrder(float d, bool affine) {
	const uint32_t o = depthOrder(d);
	return affine ? ~o : o;
}

__device__ __forceinline__ unsigned long long depthOnlyKey(float d, bool affine, uint32_t priority) {
	return ((unsigned long long)depthOnlyOrder(d, affine) << 32) | (unsigned long long)((priority << 1) | (__float_as_uint(d) >> 31));
}

// The depth a key holds.
__device__ __forceinline__ float depthOfKey(unsigned long long key, bool affine) {
	uint32_t o = (uint32_t)(key >> 32);
	if (affine) o = ~o;
	const uint32_t u = (o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o;
	return __uint_as_float(u == 0u ? (((uint32_t)key & 1u) << 31) : u);
}

template <int TW, int TH> struct DepthLds {
	static constexpr int32_t NT = TW * TH / 4;
	static constexpr int32_t CHUNK = 32;   // commands staged at once
	static constexpr int32_t LIST = 128;   // commands sorted per round (longer lists take more rounds)
	int32_t list[LIST];
	unsigned long long keys[TW * TH];
	TriangleRows tr[CHUNK];
	Command command[CHUNK];
	int32_t rowFirst[CHUNK];
	int32_t rowStart[CHUNK + 1];
	int32_t roundInfo[4];
	int32_t slot;
};

template <int TW, int TH>
__device__ void depthTile(const FrameDev &f, int32_t tile, DepthLds<TW, TH> &s) {
	using S = DepthLds<TW, TH>;
	constexpr int32_t NT = S::NT, NP = TW * TH, CHUNK = S::CHUNK;
	const int32_t n = f.tileCount[tile];
	const int32_t ci = findSegment(f.canvasTileEnd, f.canvasCount, tile);
	const CanvasDev cv = f.canvases[ci];
	const int32_t local = tile - cv.tileBase;
	const int32_t tileX0 = (local % cv.tilesX) * TW;
	const int32_t tileY0 = (local / cv.tilesX) * TH;
	const int32_t t = threadIdx.x;
	const int32_t *src = tileListOf(f, tile);
	// One projection kind per depth-only frame (one model, one camera).
	const bool affine = f.tasks[0].camera.perspective == 0;

	for (int32_t p = t; p < NP; p += NT) {
		const int32_t x = tileX0 + p % TW, y = tileY0 + p / TW;
		const float d = (x < cv.width && y < cv.height) ? cv.depth[(size_t)y * cv.depthStride + x] : 0.0f;
		s.keys[p] = d != d ? ~0ull : depthOnlyKey(d, affine, DEPTH_HELD_PRIORITY);
	}

	int32_t last = -1;
	int32_t done = 0;
	while (done < n) {
		const int32_t take = nextRound<NT, S::LIST>(src, n, done, last, s.list, s.roundInfo, (int32_t *)s.tr);
		for (int32_t c0 = 0; c0 < take; c0 += CHUNK) {
			const int32_t cn = take - c0 < CHUNK ? take - c0 : CHUNK;
			stageToLds<NT>(s.tr, (const uint8_t *)f.triangleRows, s.list, c0, cn);
			stageToLds<NT>(s.command, (const uint8_t *)f.commands, s.list, c0, cn);
			stageWait();
			__syncthreads();
			// Each command's rows inside the tile and inside the canvas, and their prefix.
			if (t < 64) {
				int32_t first = 0, count = 0;
				if (t < cn) {
					const int32_t bottom = tmin(tmin(s.tr[t].alB, cv.height) - tileY0, TH);
					first = tmin(tmax(s.tr[t].alT - tileY0, 0), TH);
					count = tmax(bottom - first, 0);
				}
				int32_t x = count;
#pragma unroll
				for (int32_t offset = 1; offset < 64; offset <<= 1) {
					const int32_t y = __shfl_up(x, offset, 64);
					if (t >= offset) x += y;
				}
				if (t < cn) {
					s.rowFirst[t] = first;
					s.rowStart[t] = x - count;
				}
				if (t == cn - 1) s.rowStart[cn] = x;
			}
			__syncthreads();
			const int32_t rowItems = s.rowStart[cn];
			for (int32_t it = t; it < rowItems; it += NT) {
				const int32_t j = segmentOf(s.rowStart, cn, it);
				const int32_t y = tileY0 + s.rowFirst[j] + (it - s.rowStart[j]);
				const RowInterval row = triangleRow(s.tr[j], y);
				const int32_t x1 = tmin(row.right, tileX0 + TW);
				if (row.left >= x1 || row.right <= tileX0) continue;
				const Projection &pl = s.command[j].plane;
				const float dx = pl.dx.x;
				float value = weightAtPixel(pl, row.left, y).x;
				int32_t x = row.left;
#pragma clang loop unroll(disable)
				for (; x < tileX0; x++) value += dx;
				const uint32_t priority = DEPTH_HELD_PRIORITY - 1u - (uint32_t)(done + c0 + j);
				unsigned long long *key = &s.keys[(y - tileY0) * TW + (x - tileX0)];
#pragma clang loop unroll(disable)
				for (; x < x1; x++) {
					if (value == value) atomicMax(key, depthOnlyKey(value, affine, priority));
					value += dx;
					key++;
				}
			}
			__syncthreads();
		}
		done += take;
		if (take == 0) break;
	}

	for (int32_t p = t; p < NP; p += NT) {
		const unsigned long long key = s.keys[p];
		if (key == ~0ull || (uint32_t)key >> 1 == DEPTH_HELD_PRIORITY) continue;
		const int32_t x = tileX0 + p % TW, y = tileY0 + p / TW;
		if (x >= cv.width || y >= cv.height) continue;
		cv.depth[(size_t)y * cv.depthStride + x] = depthOfKey(key, affine);
	}
	if (f.selfClean && t == 0) f.tileCount[tile] = 0;  // read by this workgroup alone, long before
}

template <int TW, int TH>
__global__ void __launch_bounds__(TW * TH / 4) k_raster_depth(FrameDev f) {
	__shared__ DepthLds<TW, TH> s;
	reportCounters(f);
	resetNextCounters(f);
	if (f.counters[2]) return;  // an earlier stage ran out of room: leave the canvas untouched
	forEachQueuedTile(f, 0, &s.slot, [&](int32_t tile) { depthTile<TW, TH>(f, tile, s); });
}

template __global__ void k_raster_depth<16, 16>(FrameDev);
template __global__ void k_raster_depth<32, 16>(FrameDev);
template __global__ void k_raster_depth<32, 32>(FrameDev);

// Orders one wave's LDS writes before its later reads of what other lanes of the wave wrote.
__device__ __forceinline__ void waveSync() {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The adjoint of the differentiable forward with visibility fixed: dL/dcolour of each drawn pixel goes
// into the four bilinear texels and the three corners' RGB multipliers with float atomics, through the
// weights of the (command, lane) that drew it.
//
// The forward leaves those weights in a record per drawn pixel.  Deriving them again -- two exact rows
// and the weight chain per pixel pair, from 208 bytes of command gathered per lane -- was the larger
// part of the kernel and kept it at three waves per SIMD.  A record counts only with the pixel's own
// id and the number of the last forward; any other pixel (an id written by the caller, a canvas kept
// from an earlier forward) raises a flag and is left to the DERIVE form, launched next, which ends at
// once without the flag and otherwise derives the weights of those pixels as before.
//
// Workgroups pull bands of 32x32-pixel regions (all regions of all views, whatever the forward's tile
// shape) from a queue until it is empty.  A thread takes two horizontally adjacent pixels: drawn by the
// same command they share one set of multiplier terms, and with the same four texels one set of taps.
// The multiplier gradients of the pixels of one command are first added up in LDS (a small
// open-addressed table of the region's commands), so a region makes one global atomic per (command,
// corner, channel) instead of one per pixel; commands beyond the table's room add theirs directly.
// Texture gradients are gathered the same way per texel where neighbouring pixels share their taps (a
// magnified texture); other taps, and those that find no room, are staged per wave in LDS and added with
// one lane per channel, so that one atomic instruction covers the four channels of 16 texels
// (L2 serves float atomics per cache line and request: four channels in one request instead
// of four requests).
//
// The tables add in 64 bits: an LDS float add (ds_add_f32) takes three cycles per active lane whatever
// the addresses, 192 for a full wave, where the double add takes 8 to 32 as the addresses' banks allow.
// Four of them per tap were 150 us of the 8-view fit's 460.
constexpr int32_t BACKWARD_SLOTS = 128, BACKWARD_PROBES = 16;
constexpr int32_t TEXEL_COLUMNS_LOG2 = 4, TEXEL_ROWS = 16, TEXEL_SLOTS = TEXEL_ROWS << TEXEL_COLUMNS_LOG2;
constexpr int32_t POINT_SLOTS_LOG2 = 8, POINT_SLOTS = 1 << POINT_SLOTS_LOG2, POINT_PROBES = 16;

// One pixel's share of the adjoint: its command (-1: none), the corners' points, its bilinear
// taps, dL/dtexel per channel before the tap weights, and dL/dmultiplier per corner and channel.
struct AdjointTerms {
	int32_t c;
	int32_t point[3];
	uint32_t texel[4];
	float weight[4];
	float gt[4];
	float mul[9];
};

// The second and third corner's weights of lane `lane` of the command's quad over pixel (x, y), by the
// forward's own rows and weight stepping; touches is 0 when the command does not touch the quad.
struct DerivedWeights { float wb, wc; int32_t touches; };
__device__ __forceinline__ DerivedWeights derivedWeights(const Command *commands, const TriangleRows *rows, int32_t c, int32_t lane,
                                                         int32_t x, int32_t y, int32_t canvasHeight) {
	const Command cmd = commands[c];
	const int32_t py = y & ~1;
	QuadEval e;
	if (!evalQuad(cmd, triangleRow(rows[c], py), triangleRow(rows[c], py + 1), x & ~1, py, canvasHeight, e)) return DerivedWeights{0.0f, 0.0f, 0};
	float wa[4], b[4], w[4];
	for (int l = 0; l < 4; l++) laneWeights(e, l, (cmd.flags & 1) != 0, wa[l], b[l], w[l]);
	return DerivedWeights{pick4(b, lane), pick4(w, lane), 1};
}

// heads: the queue heads of the two forms, then the flag.
template <bool DERIVE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DERIVE ? 2 : 4, DERIVE ? 2 : 4))) k_backward(FrameDev f, int32_t *heads) {
	if (DERIVE && f.diffRecords && heads[2] == 0) return;
	__shared__ int32_t unitLds;
	__shared__ int32_t slotCommand[BACKWARD_SLOTS];
	__shared__ double slotGrad[9][BACKWARD_SLOTS];
	__shared__ int32_t texelKey[TEXEL_SLOTS];
	__shared__ double texelGrad[4][TEXEL_SLOTS];
	__shared__ int32_t stageTexel[256 * 4];
	__shared__ float4 stageGrad[256 * 4];
	static_assert(POINT_SLOTS <= 256 * 4 && POINT_SLOTS * 3 * sizeof(double) <= sizeof(stageGrad), "the points' table fits the stage");
	const int32_t t = (int32_t)threadIdx.x;
	const int32_t forward = f.diffRecords ? *f.forwardNumber : 0;
	bool unknown = false;  // a pixel of this thread is left to the DERIVE form
	const uint32_t commandCount = DERIVE ? (uint32_t)f.counters[0] : 0u;

	// One of the four taps of a pixel into the region's texel table; false when another texel has its place.
	auto addToTable = [&](int32_t texel, const float4 &value) -> bool {
		const int32_t i = (((texel >> f.ftexLog2w) & (TEXEL_ROWS - 1)) << TEXEL_COLUMNS_LOG2) | (texel & ((1 << TEXEL_COLUMNS_LOG2) - 1));
		// Most taps find their texel there already: a plain read, which lanes with one address share.
		if (((volatile int32_t *)texelKey)[i] != texel) {
			const int32_t old = atomicCAS(&texelKey[i], -1, texel);
			if (old != -1 && old != texel) return false;
		}
		unsafeAtomicAdd(&texelGrad[0][i], (double)value.x);
		unsafeAtomicAdd(&texelGrad[1][i], (double)value.y);
		unsafeAtomicAdd(&texelGrad[2][i], (double)value.z);
		unsafeAtomicAdd(&texelGrad[3][i], (double)value.w);
		return true;
	};
	// The taps of a thread's two pixels: the upper two of each, then the lower two.  same: both pixels
	// hit the same texels, and the left one's taps carry the right one's share.  What the table does
	// not take is staged in the order of the columns, so that one instruction adds the four channels
	// of 16 taps of eight neighbouring pixels and one texel row: as few L2 requests as they have
	// lines.  Every lane of the wave calls it.
	auto addTaps = [&](const AdjointTerms &P, const AdjointTerms &Q, bool any, bool second, bool same, bool table) {
		const int32_t lane = t & 63, ch = lane & 3, waveBase = (t & ~63) * 4;
#pragma unroll
		for (int row = 0; row < 2; row++) {
			bool staged = false;
#pragma unroll
			for (int k = 0; k < 4; k++) {
				const AdjointTerms &T = k < 2 ? P : Q;
				const int tap = row * 2 + (k & 1);
				const float other = k < 2 && same ? Q.weight[tap] : 0.0f;
				bool due = (k < 2 ? any : second) && !(T.weight[tap] == 0.0f && other == 0.0f);
				float4 value;
				value.x = T.gt[0] * T.weight[tap] + (k < 2 && same ? Q.gt[0] * other : 0.0f);
				value.y = T.gt[1] * T.weight[tap] + (k < 2 && same ? Q.gt[1] * other : 0.0f);
				value.z = T.gt[2] * T.weight[tap] + (k < 2 && same ? Q.gt[2] * other : 0.0f);
				value.w = T.gt[3] * T.weight[tap] + (k < 2 && same ? Q.gt[3] * other : 0.0f);
				if (due && table && addToTable((int32_t)T.texel[tap], value)) due = false;
				stageTexel[t * 4 + k] = due ? (int32_t)T.texel[tap] : -1;
				if (due) stageGrad[t * 4 + k] = value;
				staged = staged || due;
			}
			if (__any(staged)) {
				// The stage is the wave's own, so a wave-scope barrier orders its writes and reads.
				waveSync();
#pragma unroll 4
				for (int32_t r = 0; r < 16; r++) {
					const int32_t e = waveBase + r * 16 + (lane >> 2);
					const int32_t to = stageTexel[e];
					if (to >= 0) unsafeAtomicAdd(f.gradTexture + (size_t)to * 4 + ch, ((const float *)stageGrad)[e * 4 + ch]);
				}
			}
			waveSync();
		}
	};
	auto addMultipliers = [&](const AdjointTerms &P) {
		int32_t slot = -1;
		const int32_t h = (int32_t)(((uint32_t)P.c * 2654435761u) >> 25);
		for (int32_t k = 0; k < BACKWARD_PROBES; k++) {
			const int32_t i = (h + k) & (BACKWARD_SLOTS - 1);
			int32_t old = ((volatile int32_t *)slotCommand)[i];
			if (old == -1) old = atomicCAS(&slotCommand[i], -1, P.c);
			if (old == -1 || old == P.c) {
				slot = i;
				break;
			}
		}
#pragma unroll
		for (int c3 = 0; c3 < 3; c3++)
#pragma unroll
			for (int ch = 0; ch < 3; ch++) {
				if (slot >= 0) unsafeAtomicAdd(&slotGrad[c3 * 3 + ch][slot], (double)P.mul[c3 * 3 + ch]);
				else unsafeAtomicAdd(f.gradMultipliers + P.point[c3] * 3 + ch, P.mul[c3 * 3 + ch]);
			}
	};

	const int32_t rows = ADJOINT_REGION / f.regionBands;
	while (true) {
		if (t == 0) unitLds = atomicAdd(&heads[DERIVE ? 1 : 0], 1);
		for (int32_t i = t; i < BACKWARD_SLOTS; i += 256) slotCommand[i] = -1;
		for (int32_t i = t; i < BACKWARD_SLOTS * 9; i += 256) (&slotGrad[0][0])[i] = 0.0;
		for (int32_t i = t; i < TEXEL_SLOTS; i += 256) texelKey[i] = -1;
		for (int32_t i = t; i < TEXEL_SLOTS * 4; i += 256) (&texelGrad[0][0])[i] = 0.0;
		__syncthreads();
		const int32_t unit = __builtin_amdgcn_readfirstlane(unitLds);
		if (unit >= f.regionTotal * f.regionBands) break;
		const int32_t region = unit / f.regionBands, band = unit % f.regionBands;
		const int32_t ci = findSegment(f.canvasRegionEnd, f.canvasCount, region);
		const CanvasDev &cv = f.canvases[ci];
		const int32_t local = region - (ci > 0 ? f.canvasRegionEnd[ci - 1] : 0), across = adjointRegions(cv.width);
		const int32_t x0 = (local % across) * ADJOINT_REGION, y0 = (local / across) * ADJOINT_REGION + band * rows;
		const int32_t commandBase = f.canvasCommandBase[ci];
		for (int32_t item = t; item < ADJOINT_REGION / 2 * rows; item += 256) {
			const int32_t x = x0 + 2 * (item % (ADJOINT_REGION / 2)), y = y0 + item / (ADJOINT_REGION / 2);
			AdjointTerms a[2];
			float weightB[2], weightC[2];
#pragma unroll
			for (int i = 0; i < 2; i++) {
				a[i].c = -1;
				if (x + i >= cv.width || y >= cv.height) continue;
				const int32_t id = cv.visibility[(size_t)y * cv.diffStride + x + i];
				if (id < 0) continue;
				const int32_t c = (int32_t)((uint32_t)(id >> 2) + (uint32_t)commandBase);
				bool known = false;
				if (f.diffRecords) {
					const DiffRecord rec = f.diffRecords[cv.recordBase + (int64_t)y * cv.width + x + i];
					known = rec.id == id && rec.forward == forward;
					weightB[i] = rec.wb;
					weightC[i] = rec.wc;
				}
				if (!DERIVE) {
					unknown = unknown || !known;
					if (!known) continue;
				} else {
					// An id that a forward before the last one left, or the caller, may name no command: of a
					// view that the last forward drew nothing in (its commandBase is unset), or of more commands.
					if (known || (uint32_t)c >= commandCount) continue;
					const DerivedWeights derived = derivedWeights(f.commands, f.triangleRows, c, id & 3, x + i, y, cv.height);
					if (!derived.touches) continue;
					weightB[i] = derived.wb;
					weightC[i] = derived.wc;
				}
				a[i].c = c;
			}
#pragma unroll
			for (int i = 0; i < 2; i++) {
				AdjointTerms &o = a[i];
				const int32_t c = o.c;
				if (c < 0) continue;
				const size_t p = (size_t)y * cv.diffStride + x + i;
				const float wbw = weightB[i], wc = weightC[i], wa = 1.0f - (wbw + wc);
				const float4 g = *(const float4 *)(cv.gradColor + p * 4);
				const DiffInputs d = f.diffInputs[c];
				const float u = interp(d.u, wa, wbw, wc), v = interp(d.v, wa, wbw, wc);
				const BilinearTaps taps = bilinearTaps(f.ftexLog2w, f.ftexLog2h, u, v);
				float tx[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
				for (int k = 0; k < 4; k++) {
					const float4 texel = *(const float4 *)(f.ftexTexels + (size_t)taps.index[k] * 4);
					tx[0] += taps.weight[k] * texel.x;
					tx[1] += taps.weight[k] * texel.y;
					tx[2] += taps.weight[k] * texel.z;
					tx[3] += taps.weight[k] * texel.w;
				}
				const float w3[3] = {wa, wbw, wc};
				float mixed[3];
#pragma unroll
				for (int ch = 0; ch < 3; ch++)
					mixed[ch] = wa * multiplier(f, d.point[0], ch) + wbw * multiplier(f, d.point[1], ch) + wc * multiplier(f, d.point[2], ch);
#pragma unroll
				for (int c3 = 0; c3 < 3; c3++) o.point[c3] = d.point[c3];
#pragma unroll
				for (int k = 0; k < 4; k++) {
					o.texel[k] = taps.index[k];
					o.weight[k] = taps.weight[k];
				}
				o.gt[0] = g.x * mixed[0];
				o.gt[1] = g.y * mixed[1];
				o.gt[2] = g.z * mixed[2];
				o.gt[3] = g.w;
				const float gm[3] = {g.x * tx[0], g.y * tx[1], g.z * tx[2]};
#pragma unroll
				for (int c3 = 0; c3 < 3; c3++)
#pragma unroll
					for (int ch = 0; ch < 3; ch++) o.mul[c3 * 3 + ch] = gm[ch] * w3[c3];
			}
			const bool v0 = a[0].c >= 0, v1 = a[1].c >= 0;
			if (f.gradTexture) {
				bool same = v0 && v1;
#pragma unroll
				for (int k = 0; k < 4; k++) same = same && a[0].texel[k] == a[1].texel[k];
				// The table pays where a pair's taps overlap: the right pixel starts at a texel of the
				// left one's, as in most of the wave's pairs of a magnified texture.
				const bool near = v0 && v1 && (a[1].texel[0] == a[0].texel[0] || a[1].texel[0] == a[0].texel[1] || a[1].texel[0] == a[0].texel[2] ||
				                               a[1].texel[0] == a[0].texel[3] || a[0].texel[0] == a[1].texel[1] || a[0].texel[0] == a[1].texel[2]);
				const bool table = 2 * __popcll(__ballot(near)) >= __popcll(__ballot(v0 && v1));
				AdjointTerms first = a[1];
				if (v0) first = a[0];
				addTaps(first, a[1], v0 || v1, v0 && v1 && !same, same, table);
			}
			if (f.gradMultipliers) {
				if (v0 && v1 && a[0].c == a[1].c) {
#pragma unroll
					for (int m = 0; m < 9; m++) a[0].mul[m] += a[1].mul[m];
					addMultipliers(a[0]);
				} else {
					if (v0) addMultipliers(a[0]);
					if (v1) addMultipliers(a[1]);
				}
			}
		}
		__syncthreads();
		if (f.gradTexture)
			for (int32_t i = t; i < TEXEL_SLOTS * 4; i += 256) {
				const int32_t texel = texelKey[i >> 2];
				if (texel >= 0) unsafeAtomicAdd(f.gradTexture + (size_t)texel * 4 + (i & 3), (float)texelGrad[i & 3][i >> 2]);
			}
		if (f.gradMultipliers) {
			// The points' table lies in the stage, which no wave uses before the next region.
			int32_t *pointKey = stageTexel;
			double *pointGrad = (double *)stageGrad;
			for (int32_t i = t; i < POINT_SLOTS; i += 256) pointKey[i] = -1;
			for (int32_t i = t; i < POINT_SLOTS * 3; i += 256) pointGrad[i] = 0.0;
			__syncthreads();
			for (int32_t i = t; i < BACKWARD_SLOTS * 3; i += 256) {
				const int32_t slot = i / 3, corner = i % 3;
				if (slotCommand[slot] < 0) continue;
				const int32_t point = f.diffInputs[slotCommand[slot]].point[corner];
				const int32_t h = (int32_t)(((uint32_t)point * 2654435761u) >> (32 - POINT_SLOTS_LOG2));
				int32_t at = -1;
				for (int32_t q = 0; q < POINT_PROBES; q++) {
					const int32_t k = (h + q) & (POINT_SLOTS - 1);
					const int32_t old = atomicCAS(&pointKey[k], -1, point);
					if (old == -1 || old == point) {
						at = k;
						break;
					}
				}
				for (int ch = 0; ch < 3; ch++) {
					const double grad = slotGrad[corner * 3 + ch][slot];
					if (at >= 0) unsafeAtomicAdd(&pointGrad[at * 3 + ch], grad);
					else unsafeAtomicAdd(f.gradMultipliers + point * 3 + ch, (float)grad);
				}
			}
			__syncthreads();
			for (int32_t i = t; i < POINT_SLOTS * 3; i += 256) {
				const int32_t point = pointKey[i / 3];
				if (point >= 0) unsafeAtomicAdd(f.gradMultipliers + point * 3 + i % 3, (float)pointGrad[i]);
			}
		}
		__syncthreads();
	}
	if (!DERIVE && unknown) atomicOr(&heads[2], 1);
}

template __global__ void k_backward<false>(FrameDev, int32_t *);
template __global__ void k_backward<true>(FrameDev, int32_t *);

// The start of a frame: zeroed counters, tile counts and fill cursors, unset canvas command bases
// and, for differentiable frames, the next forward number.
__global__ void k_frame_begin(FrameDev f) {
	const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < COUNTERS) f.counters[i] = 0;
	if (i < 2 * f.tileTotal + 1) f.tileCount[i] = 0;
	if (i < f.canvasCount) f.canvasCommandBase[i] = 0x7FFFFFFF;
	if (i == 0 && f.forwardNumber) f.forwardNumber[0]++;
}

// renderer_occludeFromExistingTriangles (rendererAPI.cpp:241-258): the Solid draw commands of
// every task given so far lower the grid under their hulls.  One thread per fan triangle.
__global__ void __launch_bounds__(256) k_occlude_existing(FrameDev f) {
	__shared__ ClipPolygon clipPolys[256 / 64];
	const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
	if (g >= f.fanTotal) return;
	const int32_t ti = findSegment(f.taskFanEnd, f.taskCount, g);
	bool single;
	(void)setupTriangle<SETUP_OCCLUDE>(f, ti, loadCorners(f, g, ti), &clipPolys[threadIdx.x >> 6], &single);
}

// renderer_occludeFromTopRows (rendererAPI.cpp:403-474), one thread per cell: the first row of
// the cell's pixel rows, over the columns the reference's scan gives that cell (it starts one
// column early after the first cell and stops at the canvas width), reduced to the farthest
// depth -- 1 / the smallest inverse depth for a perspective camera, the largest depth for an
// orthogonal one -- which replaces the cell's depth if nearer.
__global__ void k_occlude_top_rows(const float *depth, int32_t width, int32_t height, int32_t stride, float *grid, int32_t gridW,
                                   int32_t gridH, int32_t perspective) {
	const int32_t cell = blockIdx.x * blockDim.x + threadIdx.x;
	if (cell >= gridW * gridH) return;
	const int32_t gx = cell % gridW, gy = cell / gridW;
	const int32_t y = gy * OCCLUSION_CELL;
	if (y >= height) return;
	const int32_t x0 = gx == 0 ? 0 : tmin(gx * OCCLUSION_CELL - 1, width);
	const int32_t x1 = tmin(gx * OCCLUSION_CELL + OCCLUSION_CELL - 1, width);
	const float *row = depth + (size_t)y * stride;
	float farthest;
	if (perspective) {
		float smallestInverse = __builtin_huge_valf();
		for (int32_t x = x0; x < x1; x++)
			if (row[x] < smallestInverse) smallestInverse = row[x];
		farthest = 1.0f / smallestInverse;
	} else {
		farthest = 0.0f;
		for (int32_t x = x0; x < x1; x++)
			if (row[x] > farthest) farthest = row[x];
	}
	if (farthest < grid[cell]) grid[cell] = farthest;
}

// The side a row takes from one edge for count (n, d, L, R) inputs -- by the double form where its
// operands fit it, as the rows do, by the integers otherwise: the check of the row intervals' quotient
// against exact integer arithmetic.
__global__ void k_probe_edge_side(const int64_t *n, const int64_t *d, const int32_t *L, const int32_t *R, int32_t count, int32_t *out) {
	const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= count) return;
	const double m = d[i] < 0 ? -(double)n[i] : (double)n[i], a = fabs((double)d[i]);
	const bool fits = fabs(m) < 4503599627370496.0 && a < 4294967296.0 && (double)(float)a == a && fabs(m) < 1073741824.0 * a &&
	                  L[i] >= -65536 && L[i] <= 65536 && R[i] >= -65536 && R[i] <= 65536;
	out[i] = fits ? rowSide(m, (float)a, 1.0f / (float)a, L[i], R[i]) : edgeSide(n[i], d[i], L[i], R[i]);
}

__global__ void k_fill(int32_t *p, int32_t n, int32_t value) {
	int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) p[i] = value;
}

// image_fill of every canvas (colour and depth), one thread per pixel of the frame's tiles.
__global__ void k_clear_canvases(FrameDev f, uint32_t color, float depth) {
	const int32_t tile = blockIdx.x;
	if (tile >= f.tileTotal) return;
	const int32_t ci = findSegment(f.canvasTileEnd, f.canvasCount, tile);
	const CanvasDev cv = f.canvases[ci];
	const int32_t local = tile - cv.tileBase;
	const int32_t x0 = (local % cv.tilesX) * f.tileW, y0 = (local / cv.tilesX) * f.tileH;
	for (int32_t i = threadIdx.x; i < f.tileW * f.tileH; i += blockDim.x) {
		int32_t x = x0 + i % f.tileW, y = y0 + i / f.tileW;
		if (x >= cv.width || y >= cv.height) continue;
		if (cv.color) cv.color[(size_t)y * cv.colorStride + x] = color;
		if (cv.depth) cv.depth[(size_t)y * cv.depthStride + x] = depth;
		if (cv.diffColor) {
			size_t p = (size_t)y * cv.diffStride + x;
			*(float4 *)(cv.diffColor + p * 4) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
			cv.visibility[p] = -1;
		}
	}
}

// ---------------------------------------------------------------------------------------
// texture_generatePyramid on the GPU: one level from the next larger, truncating the mean
// of each 2x2 block per channel (textureAPI.cpp:44-63).
// ---------------------------------------------------------------------------------------
__global__ void k_downsample(uint32_t *texels, TextureDesc t, uint32_t targetLevel) {
	uint32_t w = 1u << (t.log2w - targetLevel), h = 1u << (t.log2h - targetLevel);
	uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= w * h) return;
	uint32_t x = i % w, y = i / w;
	uint32_t src = targetLevel - 1;
	uint32_t a = texels[pixelOffset(t, x * 2, y * 2, src)];
	uint32_t b = texels[pixelOffset(t, x * 2 + 1, y * 2, src)];
	uint32_t c = texels[pixelOffset(t, x * 2, y * 2 + 1, src)];
	uint32_t d = texels[pixelOffset(t, x * 2 + 1, y * 2 + 1, src)];
	uint32_t out = 0;
	for (uint32_t ch = 0; ch < 32; ch += 8) {
		uint32_t sum = ((a >> ch) & 255u) + ((b >> ch) & 255u) + ((c >> ch) & 255u) + ((d >> ch) & 255u);
		out |= (sum / 4u) << ch;
	}
	texels[pixelOffset(t, x, y, targetLevel)] = out;
}

}  // namespace dfpsr
