// rgl_inorder.h — the in-order tile path of the gfx950 rgl pipeline.
//
// Frames whose state the order-independent visibility keys cannot express
// are drawn here as the reference draws every tile (GPU::DrawImpl,
// rglv_gpu.cxx:263-432): each tile walks its commands in submission order.
// That covers alpha blending, the scissor test, depth test or depth writes
// off, GL_EQUAL, draws with different depth functions, and clears and stores
// between draws (a depth-only clear for a shadow pass, a store followed by
// more drawing).
//
//   k_tile_order  one workgroup per tile: the tile's (triangle, tile) pairs,
//                 inline (set up here) and clipped (setup records), sorted by
//                 submission slot and written in that order as records with
//                 their draw's state and vertices, and per region of the tile
//                 a bit per sorted record that can touch it.
//   k_inorder     one wave per 8 x 8-pixel region of a tile, one lane per
//                 pixel: the pixel's colour, depth and primitive id stay in
//                 registers while the wave steps through the region's
//                 triangles (64 at a time) and the frame commands in slot
//                 order, applying TriangleProgram::Render
//                 (rglv_gpu_impl.hxx:166-222): coverage, scissor, early or
//                 late depth test, depth write, shading, alpha blend, masked
//                 colour store.
#pragma once

#include "rgl_kernels.h"

namespace rgl {

// A frame command that every tile executes at one point of the submission
// order: CLEAR and the STORE_* commands that GPU::BinImpl broadcasts to all
// tiles (rglv_gpu.cxx:139-191).  pos is the first visibility slot it
// precedes: the triangles drawn before it have smaller slots.
enum FrameOpKind { kOpClear = 0, kOpStoreColor = 1, kOpStoreDepth = 2, kOpStorePrim = 3,
	kOpStoreColorFP = 4,      // CMD_STORE_COLOR_FULL_LINEAR_FP: RGBA float pixels (A = 0)
	kOpStoreColorHalf = 5,    // CMD_STORE_COLOR_HALF_LINEAR_FP: 2 x 2 box average (Downsample)
	kOpStoreColorQuads = 6 }; // CMD_STORE_COLOR_FULL_QUADS_FP: the quad-swizzled qfloat4 canvas
struct alignas(16) FrameOp {
	uint32_t pos;
	int kind;
	int bits;            // clear: GL_COLOR_BUFFER_BIT (1) | GL_DEPTH_BUFFER_BIT (2)
	int gamma;           // store colour: sRGB (1) or to_tc_basic (0)
	float color[4];      // clear colour (alpha: RB_RGBAF32's fourth channel)
	float depth;         // clear depth
	int post;            // store colour: post program (1 default, 2 exposure, 3 IQ)
	float exposure;
	int stride;          // float stores: the target's row stride, in pixels (quads for kOpStoreColorQuads)
	int attach;          // float stores: the colour attachment type (the quad store's alpha source)
	int pad[3];
	void* ptr;           // store target; truecolor, depth and id stores have row stride = the frame's width
};

// the in-order frames of a batch: their first k_tile_order block (one per
// tile) and first k_inorder block (one per region of a tile)
struct alignas(16) IoFrame {
	int frame;
	int tileStart;
	int blockStart;
	int regionsX, regionsY;
	int pad[3];
};

// colour attachment types (rglv_gl.hxx RB_COLOR_DEPTH, RB_RGBF32)
constexpr int kAttachColorDepth = 0, kAttachRGBF32 = 1;

constexpr int kSortCap = 4096;       // records a tile sorts in LDS in one piece
constexpr int kSortThreads = 1024;   // k_tile_order workgroup
constexpr int kRegionDim = 8;        // k_inorder region: 8 x 8 pixels, a lane each
constexpr int kIoThreads = kRegionDim * kRegionDim;
static_assert(kIoThreads == 64, "a region is one wave, its record masks one word per 64 records");

__device__ inline int find_io(const IoFrame* io, int n, int blk, bool tiles) {
	int lo = 0, hi = n - 1;
	while (lo < hi) {
		const int mid = (lo + hi + 1) >> 1;
		if ((tiles ? io[mid].tileStart : io[mid].blockStart) <= blk) lo = mid; else hi = mid - 1; }
	return lo; }

// the wave's 64 keys, one per lane, in ascending order (a bitonic network)
__device__ inline unsigned long long wave_sort(unsigned long long v) {
	const uint32_t lane = threadIdx.x & 63;
#pragma unroll
	for (uint32_t k = 2; k <= 64; k <<= 1)
#pragma unroll
		for (uint32_t j = k >> 1; j > 0; j >>= 1) {
			const unsigned long long o = __shfl_xor(v, static_cast<int>(j), 64);
			const bool low = (lane & j) == 0, up = (lane & k) == 0;
			if ((low == up) ? o < v : o > v) v = o; }
	return v; }

// one merge pass over n distinct keys in sorted runs of `run` (a power of
// two): each key's place in its merged run of 2 run is its index in its own
// run plus its rank in the other.  A thread searches for two keys at a time,
// so that one's loads fill the other's latency.
__device__ inline void merge_runs(const unsigned long long* src, unsigned long long* dst, uint32_t n, uint32_t run) {
	for (uint32_t i = threadIdx.x; i < n; i += 2 * blockDim.x) {
		unsigned long long key[2];
		uint32_t other[2], len[2], rank[2] = { 0, 0 }, out[2];
#pragma unroll
		for (uint32_t k = 0; k < 2; ++k) {
			const uint32_t j = min(i + k * blockDim.x, n - 1);   // past the last key: that key again, not stored
			const uint32_t a0 = j & ~(2 * run - 1), a1 = min(a0 + run, n), b1 = min(a0 + 2 * run, n);
			const bool inA = j < a1;
			key[k] = src[j];
			other[k] = inA ? a1 : a0; len[k] = inA ? b1 - a1 : a1 - a0;
			out[k] = inA ? j : j - run; }   // the place without the other run's keys
		for (uint32_t s = run; s > 0; s >>= 1)
#pragma unroll
			for (uint32_t k = 0; k < 2; ++k) {
				const uint32_t at = rank[k] + s;
				if (at <= len[k] && src[other[k] + at - 1] < key[k]) rank[k] = at; }
#pragma unroll
		for (uint32_t k = 0; k < 2; ++k)
			if (i + k * blockDim.x < n) dst[out[k] + rank[k]] = key[k]; }}

// A tile's record as k_inorder reads it: the setup (dx31 = -(dx12 + dx23)
// and dy31 likewise, in the wrapping arithmetic of the setup), its
// triangle's vertices and its draw's fragment state, so that a region takes
// a triangle with one 64-byte load.
struct alignas(16) IoRec {
	int32_t c1, c2, c3;
	int32_t dx12, dy12, dx23, dy23;
	uint32_t minxy;       // minx | miny << 16
	float scale;
	uint32_t slot;
	uint32_t v0, v1, v2;  // vertices (bit 31 of v0: in the clipped arrays)
	uint32_t meta;        // draw | state << 8 | quads across << 16 | quads down << 24
	uint32_t prim;        // primitive id
	uint32_t pad;
};
static_assert(sizeof(IoRec) == 64 && kMaxDraws <= 256 && kMaxAnyTileDim / 2 <= 255, "four 16-byte loads; the fields of meta");
// the fragment state in IoRec::meta >> 8: depth test, depth write, depth
// function (two bits), colour write, blend, early depth test, and whether
// the program runs (its colour or its discard is used)
constexpr uint32_t kStDepthTest = 1u, kStDepthWrite = 2u, kStDepthFunc = 2, kStColor = 16u, kStBlend = 32u, kStEarlyZ = 64u, kStProgram = 128u;

__device__ inline IoRec make_io_rec(const TriSetup& r, const DrawLite* __restrict__ lite, const DrawDesc* __restrict__ draws, int nDraws,
                                    const uint4* __restrict__ tvert, const uint32_t* __restrict__ clipqOf) {
	const int di = find_draw_slot(lite, nDraws, r.slot);
	const DrawLite& dl = lite[di];
	const DrawDesc& dd = draws[di];
	const ProgramInfo info = program_info(dd.program);
	const uint32_t rel = r.slot - dl.slotBase;
	const uint32_t nTri = static_cast<uint32_t>(dl.tris) * static_cast<uint32_t>(dl.instances);
	const uint32_t srcTri = rel < nTri ? rel : (rel - nTri) / kFanMax;
	IoRec o;
	o.c1 = r.c1; o.c2 = r.c2; o.c3 = r.c3;
	o.dx12 = r.dx12; o.dy12 = r.dy12; o.dx23 = r.dx23; o.dy23 = r.dy23;
	o.minxy = static_cast<uint32_t>(r.minx & 0xffff) | (static_cast<uint32_t>(r.miny) << 16); o.scale = r.scale; o.slot = r.slot;
	if (rel < nTri) {
		const uint4 tv = tvert[dl.triBase + srcTri];
		o.v0 = tv.x; o.v1 = tv.y; o.v2 = tv.z; }
	else {   // the fan triangle's vertices (clipped_verts)
		const uint32_t v0 = clipqOf[dl.triBase + srcTri] * kClipVerts, fj = rel - nTri - srcTri * kFanMax;
		o.v0 = v0 | 0x80000000u; o.v1 = v0 + fj + 1; o.v2 = v0 + fj + 2; }
	const uint32_t st = (dd.depthTest ? kStDepthTest : 0u) | (dd.depthWrite ? kStDepthWrite : 0u) |
	                    (static_cast<uint32_t>(dd.depthFunc) << kStDepthFunc) | (dd.colorWrite ? kStColor : 0u) |
	                    (dd.blend ? kStBlend : 0u) | (info.earlyZ ? kStEarlyZ : 0u) | (dd.colorWrite || info.discard ? kStProgram : 0u);
	o.meta = static_cast<uint32_t>(di) | (st << 8) | ((static_cast<uint32_t>(r.nqx) & 0xffu) << 16) | (static_cast<uint32_t>(r.nqy) << 24);
	o.prim = dl.primBase + srcTri;
	o.pad = 0u;
	return o; }

// The word of a tile's record masks: masks[mask_word(...) + region * nb + k]
// holds a bit per record 64 k .. 64 k + 63 of the tile's sorted list (nb =
// ceil(n / 64) words per region) whose quads reach the region.  ob: the
// tile's first sorted record, blk its index among the in-order tiles;
// maxRegions: the most regions per tile of the batch's in-order frames.
// Ranges of different tiles are disjoint.
__device__ inline long long mask_word(uint32_t ob, int blk, int maxRegions) {
	return (static_cast<long long>(ob >> 6) + blk) * maxRegions; }

// A tile's records in submission order.  Keys are (slot << 32 | p), p the
// record's position in the tile (inline records first, then clipped); every
// (triangle, tile) pair has its own slot, so keys are distinct.  sorted[ob +
// k] receives the k-th record, ob = the tile's first inline + first clipped
// list position (the tiles' ranges are disjoint).  Runs of 64 are sorted in
// the lanes of a wave, then merged in LDS (up to kSortCap records, and above
// that in global memory), each pass a binary search per key: six passes of
// LDS latency for 4,096 records, where a bitonic network in LDS took 78
// passes and barriers (71 -> 31 us with tiles of up to 1,800).  With the
// pairs set up here 38.2 us; 34.5 with two keys a thread searched together
// and a record's regions from 8 + 8 ballots instead of 64.
__global__ __launch_bounds__(kSortThreads) void k_tile_order(BatchDesc b, RasterArgs a, const IoFrame* __restrict__ io, int nIo,
		const FrameDesc* __restrict__ frames, const DrawDesc* __restrict__ draws, const DrawLite* __restrict__ lite,
		const VisTile* __restrict__ tileDesc, PairLists pl, const VisRec* __restrict__ crec,
		IoRec* __restrict__ sorted, unsigned long long* __restrict__ skeys0, unsigned long long* __restrict__ skeys1,
		unsigned long long* __restrict__ masks, int maxRegions) {
	__shared__ unsigned long long s[2][kSortCap];
	const int blk = static_cast<int>(blockIdx.x);
	const IoFrame e = io[find_io(io, nIo, blk, true)];
	const FrameDesc& f = frames[e.frame];
	const int lt = blk - e.tileStart, tile = f.tileBase + lt;
	const Rect R = tile_rect(f, lt);
	const VisTile d = tileDesc[tile];
	const uint32_t n = d.ntot, ninl = d.ninl, ob = d.ib + d.cb;
	const uint32_t t = threadIdx.x, lane = t & 63;
	auto key_of = [&](uint32_t p) -> unsigned long long {
		const uint32_t slot = p < ninl ? pl.ids[d.ib + p].w : crec[d.cb + (p - ninl)].slot;
		return (static_cast<unsigned long long>(slot) << 32) | p; };
	// records c0 .. c0 + cn - 1 sorted in LDS; returns the buffer they end in
	auto sort_lds = [&](uint32_t c0, uint32_t cn) {
		for (uint32_t i0 = t & ~63u; i0 < cn; i0 += kSortThreads) {   // uniform over the wave
			const unsigned long long v = wave_sort(i0 + lane < cn ? key_of(c0 + i0 + lane) : ~0ull);
			if (i0 + lane < cn) s[0][i0 + lane] = v; }
		__syncthreads();
		int cur = 0;
		for (uint32_t run = 64; run < cn; run <<= 1, cur ^= 1) { merge_runs(s[cur], s[cur ^ 1], cn, run); __syncthreads(); }
		return cur; };
	const unsigned long long* keys;   // the tile's sorted keys
	if (n <= static_cast<uint32_t>(kSortCap)) keys = s[sort_lds(0, n)];
	else {
		unsigned long long* src = skeys0 + ob;
		unsigned long long* dst = skeys1 + ob;
		for (uint32_t c0 = 0; c0 < n; c0 += kSortCap) {
			const uint32_t cn = min(static_cast<uint32_t>(kSortCap), n - c0);
			__syncthreads();
			const unsigned long long* v = s[sort_lds(c0, cn)];
			for (uint32_t i = t; i < cn; i += kSortThreads) src[c0 + i] = v[i]; }
		__syncthreads();
		for (uint32_t run = kSortCap; run < n; run <<= 1) {
			merge_runs(src, dst, n, run);
			__syncthreads();
			unsigned long long* x = src; src = dst; dst = x; }
		keys = src; }
	// the records in order and their masks, one wave per 64: a ballot per region
	unsigned long long* const tm = masks + mask_word(ob, blk, maxRegions);
	const uint32_t nb = (n + 63) >> 6;
	for (uint32_t k = t >> 6; k < nb; k += kSortThreads / 64) {   // uniform over the wave
		int gx0 = 1, gx1 = 0, gy0 = 1, gy1 = 0;   // the regions the record's quads reach (none)
		if (64 * k + lane < n) {
			const uint32_t p = static_cast<uint32_t>(keys[64 * k + lane]);
			TriSetup r;
			if (p < ninl) {
				const uint4 id = pl.ids[d.ib + p];
				pair_setup(pl, id, pair_rect(pl, id, pl.boxes[d.ib + p], R), r); }
			else rec_setup(crec[d.cb + (p - ninl)], r);
			const int minx = r.minx - R.x0, miny = r.miny - R.y0;
			const int nqx = r.nqx, nqy = r.nqy;
			if (nqx > 0 && nqy > 0) {
				gx0 = minx / kRegionDim; gx1 = (minx + 2 * nqx - 1) / kRegionDim;
				gy0 = miny / kRegionDim; gy1 = (miny + 2 * nqy - 1) / kRegionDim; }
			sorted[ob + 64 * k + lane] = make_io_rec(r, lite, draws, b.nDraws, a.tvert, a.clipqOf); }
		// a lane per region, its word the ballots of its column and its row
		const int regions = e.regionsX * e.regionsY;
		for (int reg0 = 0; reg0 < regions; reg0 += 64) {
			const int reg = reg0 + static_cast<int>(lane), ry = reg / e.regionsX, rx = reg - ry * e.regionsX;
			unsigned long long col = 0, rowm = 0;
			for (int g = 0; g < e.regionsX; ++g) { const unsigned long long m = __ballot(gx0 <= g && g <= gx1); if (rx == g) col = m; }
			for (int g = 0; g < e.regionsY; ++g) { const unsigned long long m = __ballot(gy0 <= g && g <= gy1); if (ry == g) rowm = m; }
			if (reg < regions) tm[static_cast<long long>(reg) * nb + k] = col & rowm; }}}

// the draw's program on one lane of a quad, the vertices' varyings loaded
// with the triangle's vertex ids
struct ShadeFrag {
	const DrawDesc& d; const TriSetup& t; const TriVerts& tr; const float* vary;
	int kx, ky, lane, h; float* col; float depth; bool keep;
	template <class P> __device__ void run() {
		typename ShadeOne<P>::Vary vy;
		ShadeOne<P>::load(vary, tr, vy);
		keep = shade_lane<P>(d, t, tr, vy.v[0], vy.v[1], vy.v[2], kx, ky, lane, kRcpMantissa, col, depth, h); }};

// depth functions of the fragment state (DepthLT / DepthLE / DepthEQ,
// rglv_gpu_impl.hxx:64-74)
__device__ inline bool depth_pass(int func, float frag, float dest) {
	return func == 0 ? frag < dest : func == 1 ? frag <= dest : frag == dest; }

// the k-th (from 0) set bit of m, which has more than k
__device__ inline uint32_t select_bit(unsigned long long m, uint32_t k) {
	uint32_t at = 0;
	uint32_t w = static_cast<uint32_t>(m);
	uint32_t c = static_cast<uint32_t>(__popc(w));
	if (k >= c) { k -= c; at = 32; w = static_cast<uint32_t>(m >> 32); }
#pragma unroll
	for (uint32_t h = 16; h > 0; h >>= 1) {
		c = static_cast<uint32_t>(__popc(w & ((1u << h) - 1u)));
		if (k >= c) { k -= c; at += h; w >>= h; }}
	return at; }

// A region's triangles come 64 at a time (the set bits of its record masks,
// in order), and their (triangle, quad) pairs inside the region, at most 16
// each, in windows of 64.  Cover: each lane takes one pair and lists its
// covered fragments.  Rounds of 64 listed fragments follow.  Shade: each lane
// takes one fragment and runs the program (programs have no side effects, so
// this runs before the depth test); its bit goes into its pixel's word.
// Apply: each lane walks the set bits of its pixel, in slot order, with the
// frame's commands between them.
//
// Bound: VALU issue (the program per fragment, about 60 of its 111 us on
// 327,680 blended triangles at 1920x1080) and the two dependent fetches of a
// round (positions with varyings, texels).  The LDS is kept to 8 KB, 19 waves
// a CU, by holding one round's colours.  On the same frame: the colours of a
// whole window (12 KB) 123 us, a lane per quad in the shading, three of whose
// four lanes are often not covered, 219 us, and 16 x 16 regions that walked
// all triangles of a batch per quad and all batches of the tile 471 us.
//
// L: the programs the draws may use (a frame of one program compiles only
// that program's shading, which keeps the registers, and so the resident
// waves that hide each triangle's texture fetches, of that program alone)
template <class L>
__global__ __launch_bounds__(kIoThreads) void k_inorder(BatchDesc b, RasterArgs a, const IoFrame* __restrict__ io, int nIo,
		const FrameDesc* __restrict__ frames, const FrameOp* __restrict__ ops, const DrawDesc* __restrict__ draws,
		const DrawLite* __restrict__ lite, const VisTile* __restrict__ tileDesc, const IoRec* __restrict__ sorted,
		const unsigned long long* __restrict__ masks, int maxRegions, const uint32_t* __restrict__ order) {
	// 64 words of the region's record masks and the set bits before each
	__shared__ unsigned long long smask[64];
	__shared__ uint32_t spre[65];
	// the batch's triangles, and their pair rects in the region's quads (x0 |
	// y0 << 4 | cx << 8) and first pairs
	__shared__ IoRec stri[64];
	__shared__ uint32_t srect[64], qoff[64];
	// a window of pairs: its triangles; the covered fragments that wait to be
	// shaded (triangle | pixel of the region << 6); a round of 64 of them:
	// triangles, depths, colours, whether the program kept them, and per pixel
	// the round's fragments
	__shared__ uint8_t wtri[64];
	__shared__ uint16_t flist[64 + 256];
	__shared__ uint8_t rtri[64], rkeep[64];
	__shared__ float rfd[64];
	__shared__ float4 rcol[64];
	__shared__ unsigned long long pfrags[64];
	const int vs = a.varyStride;
	// Workgroups are dealt round-robin over the eight XCDs: runs of 64 regions
	// (a 64-pixel tile's) go to one XCD, whose L2 then reads the tile's
	// records, vertices and texels once.
	constexpr int kRun = 64 * kXcds;
	const int wg = static_cast<int>(blockIdx.x);
	const int blk = wg < static_cast<int>(gridDim.x) / kRun * kRun ? wg / kRun * kRun + (wg % kXcds) * 64 + (wg / kXcds) % 64 : wg;
	// With `order` (frames drawn in order alone, of one tile size) the tiles
	// come as the scan ordered them, the most records first in classes of
	// powers of two, so that the longest regions do not start last.
	const IoFrame e0 = io[order ? 0 : find_io(io, nIo, blk, false)];
	const int rpt = e0.regionsX * e0.regionsY;
	const int lb = blk - e0.blockStart, ltn = lb / rpt, reg = lb - ltn * rpt;
	const int tile = order ? static_cast<int>(order[ltn]) : frames[e0.frame].tileBase + ltn;
	const VisTile vt = tileDesc[tile];
	const IoFrame e = order && nIo > 1 ? io[vt.flags & 0xffu] : e0;
	const FrameDesc& f = frames[e.frame];
	const int lt = tile - f.tileBase;
	const Rect R = tile_rect(f, lt);
	const int rgy = reg / e.regionsX, rgx = reg - rgy * e.regionsX;
	const int rx0 = R.x0 + rgx * kRegionDim, ry0 = R.y0 + rgy * kRegionDim;
	if (rx0 >= R.x1 || ry0 >= R.y1) return;   // beyond the target (uniform): no quad starts here
	const int t = static_cast<int>(threadIdx.x);
	// this lane's pixel: lane l = (l & 1, l >> 1) of quad `quad` at (qx, qy)
	const int l = t & 3, quad = t >> 2;
	const int qx = rx0 + 2 * (quad & 3), qy = ry0 + 2 * (quad >> 2);
	const int x = qx + (l & 1), y = qy + (l >> 1);
	const bool onScreen = x < R.x1 && y < R.y1;
	const bool quadOnScreen = qx < R.x1 && qy < R.y1;
	// the tile buffers start zeroed (the oracle's convention for a tile not
	// yet cleared; the reference leaves the previous tile's contents)
	float cr = 0.0F, cg = 0.0F, cb = 0.0F, dz = 0.0F;
	float ca = 0.0F;   // RB_RGBAF32's alpha: set by clears, never drawn
	uint32_t pid = 0xffffffffu;
	uint32_t frags = 0;
	const uint32_t n = vt.ntot, ob = vt.ib + vt.cb;
	uint32_t opi = static_cast<uint32_t>(f.opBase);
	const uint32_t ope = static_cast<uint32_t>(f.opBase + f.nOps);
	uint32_t nextOp = opi < ope ? ops[opi].pos : 0xffffffffu;   // the position of the next frame command

	// every lane of the wave runs it (the downsampling store reads a quad's lanes)
	auto apply_op = [&](const FrameOp& op) {
		if (op.kind == kOpClear) {
			if (op.bits & 1) { cr = op.color[0]; cg = op.color[1]; cb = op.color[2]; ca = op.color[3]; pid = 0xffffffffu; }
			if (op.bits & 2) dz = op.depth; }
		else if (op.kind == kOpStoreColorHalf) {
			// Downsample (rglr_algorithm.cxx:118-165): one output per quad whose
			// top-left pixel lies in the tile rect (the reference's loops step
			// 2 x 2 over the rect), the transposed quad's pixels summed in lane
			// order, times 1/4; alpha 0
			auto mean = [&](float v) {
				const float v1 = __shfl(v, (t & ~3) + 1, 64), v2 = __shfl(v, (t & ~3) + 2, 64), v3 = __shfl(v, (t & ~3) + 3, 64);
				return (((v + v1) + v2) + v3) * 0.25F; };
			const float r = mean(cr), g = mean(cg), bl = mean(cb);
			const float z = ((0.0F + 0.0F) + 0.0F) + 0.0F;
			if (quadOnScreen && l == 0)
				static_cast<float4*>(op.ptr)[static_cast<long long>(qy >> 1) * op.stride + (qx >> 1)] = make_float4(r, g, bl, z * 0.25F); }
		else if (op.kind == kOpStoreColorQuads) {
			// Copy to a QFloat4Canvas (rglr_algorithm.cxx:320-368): alpha 1
			// from RB_RGBF32, the fourth channel (RB_COLOR_DEPTH: the depth)
			// otherwise
			if (!quadOnScreen) return;
			float* o = static_cast<float*>(op.ptr) + 16 * (static_cast<long long>(qy >> 1) * op.stride + (qx >> 1)) + l;
			o[0] = cr; o[4] = cg; o[8] = cb;
			o[12] = op.attach == kAttachRGBF32 ? 1.0F : op.attach == kAttachColorDepth ? dz : ca; }
		else {
			if (!onScreen) return;
			const long long o = static_cast<long long>(y) * f.W + x;
			if (op.kind == kOpStoreColor) {
				float c[3] = { cr, cg, cb };
				if (op.post != 1) post_shade(op.post, op.exposure, c, f.W, f.H, R.x0, R.y0, x, y);
				const uint32_t px = op.gamma
					? ((to_srgb8(c[0]) << 16) | (to_srgb8(c[1]) << 8) | to_srgb8(c[2]))
					: ((to_linear8(c[0]) << 16) | (to_linear8(c[1]) << 8) | to_linear8(c[2]));
				static_cast<uint32_t*>(op.ptr)[o] = px; }
			else if (op.kind == kOpStoreDepth) static_cast<float*>(op.ptr)[o] = dz;
			else if (op.kind == kOpStoreColorFP)   // Copy to a FloatingPointCanvas (rglr_algorithm.cxx:194-280): alpha 0
				static_cast<float4*>(op.ptr)[static_cast<long long>(y) * op.stride + x] = make_float4(cr, cg, cb, 0.0F);
			else static_cast<uint32_t*>(op.ptr)[o] = pid; }};

	// the round's fragments of this pixel (bits of todo), in submission order
	auto apply_frags = [&](unsigned long long todo) {
		while (todo) {
			const int w = __ffsll(static_cast<long long>(todo)) - 1;
			todo &= todo - 1;
			const int j = rtri[w];
			const uint32_t st = stri[j].meta >> 8;
			const float fd = rfd[w];
			const float4 c = rcol[w];
			const bool keep = rkeep[w] != 0;   // gl_triMask after ShadeFragment
			const bool pass = !(st & kStDepthTest) || depth_pass(static_cast<int>((st >> kStDepthFunc) & 3u), fd, dz);
			bool on;
			if (st & kStEarlyZ) {   // early depth test and write
				if (pass && (st & kStDepthWrite)) dz = fd;
				on = pass && keep; }
			else {
				on = keep && pass;
				if (on && (st & kStDepthWrite)) dz = fd; }
			if (on) {
				if (st & kStColor) {
					if (st & kStBlend) {   // BlendAlpha (rglv_gpu_impl.hxx:80-84)
						const float al = c.w, om = 1.0F - al;
						cr = c.x * al + cr * om;
						cg = c.y * al + cg * om;
						cb = c.z * al + cb * om; }
					else { cr = c.x; cg = c.y; cb = c.z; }}
				pid = stri[j].prim; }}};

	// one round: cnt of the listed fragments from f0 on (1 to 64), a lane each
	auto round = [&](uint32_t f0, uint32_t cnt) {
		uint32_t slot = 0xffffffffu;
		if (static_cast<uint32_t>(t) < cnt) {
			const uint32_t en = flist[f0 + static_cast<uint32_t>(t)];
			const int j = static_cast<int>(en & 63u), fl = static_cast<int>((en >> 6) & 3u), wq = static_cast<int>(en >> 8);
			const IoRec& r = stri[j];
			TriSetup ts;
			ts.c1 = r.c1; ts.c2 = r.c2; ts.dx12 = r.dx12; ts.dy12 = r.dy12; ts.dx23 = r.dx23; ts.dy23 = r.dy23;
			ts.minx = static_cast<int>(r.minxy & 0xffffu); ts.miny = static_cast<int>(r.minxy >> 16); ts.scale = r.scale;
			const int kx = (rx0 + 2 * (wq & 3) - ts.minx) >> 1, ky = (ry0 + 2 * (wq >> 2) - ts.miny) >> 1;
			const bool clipped = (r.v0 >> 31) != 0u;
			const uint32_t vi[3] = { r.v0 & 0x7fffffffu, r.v1, r.v2 };
			const float4* vp = clipped ? a.cvpos : a.vpos;
			TriVerts tr;
			tr.clipped = clipped;
#pragma unroll
			for (int i = 0; i < 3; ++i) {
				const float4 p = vp[vi[i]];
				tr.z[i] = p.z; tr.w[i] = p.w;
				tr.vary[i] = static_cast<long long>(vi[i]) * vs; }
			const uint32_t meta = r.meta;
			const DrawDesc& dd = draws[meta & 0xffu];
			float col[4] = { 0.0F, 0.0F, 0.0F, 0.0F }, fd;
			bool keep = true;
			if (meta & (kStProgram << 8)) {
				ShadeFrag sf{ dd, ts, tr, clipped ? a.cvvary : a.vvary, kx, ky, fl, f.H, col, 0.0F, true };
				dispatch_program(dd.program, sf, L{});
				fd = sf.depth; keep = sf.keep; }
			else {   // neither its colour nor its discard is used: the depth alone
				const int32_t q1 = wadd(wadd(ts.c1, wmul(kx, wmul(ts.dy12, 2))), wmul(ky, wmul(ts.dx12, 2)));
				const int32_t q2 = wadd(wadd(ts.c2, wmul(kx, wmul(ts.dy23, 2))), wmul(ky, wmul(ts.dx23, 2)));
				const int32_t e1 = wadd(q1, wadd((fl & 1) ? ts.dy12 : 0, (fl & 2) ? ts.dx12 : 0));
				const int32_t e2 = wadd(q2, wadd((fl & 1) ? ts.dy23 : 0, (fl & 2) ? ts.dx23 : 0));
				const float bx = itof(e2) * ts.scale, bz = itof(e1) * ts.scale, by = (1.0F - bx) - bz;
				fd = (bx * tr.z[0] + by * tr.z[1]) + bz * tr.z[2]; }
			rtri[t] = static_cast<uint8_t>(j);
			rkeep[t] = keep ? 1 : 0;
			rfd[t] = fd;
			rcol[t] = make_float4(col[0], col[1], col[2], col[3]);
			slot = r.slot;
			atomicOr(&pfrags[en >> 6], 1ull << t); }
		__syncthreads();
		// apply: this pixel's fragments with the frame commands between them:
		// TriangleProgram::Render's early or late depth test and depth write
		// around the program, then blend and the masked colour store.  A
		// command takes the whole wave between the fragments before and after
		// it.
		unsigned long long todo = pfrags[t];
		pfrags[t] = 0;
		const uint32_t last = __builtin_amdgcn_readlane(slot, static_cast<int>(cnt) - 1);
		while (nextOp <= last) {
			const unsigned long long before = __ballot(slot < nextOp);
			apply_frags(todo & before);
			todo &= ~before;
			apply_op(ops[opi]);
			++opi;
			nextOp = opi < ope ? ops[opi].pos : 0xffffffffu; }
		apply_frags(todo);
		__syncthreads(); };

	const uint32_t nb = (n + 63) >> 6;   // words of the region's record masks
	const unsigned long long* rm = masks + mask_word(ob, e.tileStart + lt, maxRegions) + static_cast<long long>(reg) * nb;
	pfrags[t] = 0;
	for (uint32_t k0 = 0; k0 < nb; k0 += 64) {   // 64 words, 4,096 records, at a time
		const unsigned long long mw = k0 + t < nb ? rm[k0 + t] : 0ull;
		uint32_t hits = static_cast<uint32_t>(__popcll(mw));
		for (int o = 1; o < 64; o <<= 1) {
			const uint32_t v = __shfl_up(hits, o, 64);
			if (t >= o) hits += v; }
		const uint32_t nh = __shfl(hits, 63, 64);
		if (nh == 0) continue;   // uniform
		__syncthreads();
		smask[t] = mw;
		spre[t + 1] = hits;
		if (t == 0) spre[0] = 0;
		__syncthreads();
		// the region's h-th record of these words
		auto record = [&](uint32_t h) {
			uint32_t lo = 0;   // the word with spre[lo] <= h < spre[lo + 1]
#pragma unroll
			for (uint32_t st = 32; st > 0; st >>= 1) if (spre[lo + st] <= h) lo += st;
			return sorted[ob + 64 * (k0 + lo) + select_bit(smask[lo], h - spre[lo])]; };
		// each lane's record of the next batch is loaded while this one is drawn
		IoRec rn;
		if (static_cast<uint32_t>(t) < nh) rn = record(static_cast<uint32_t>(t));
		for (uint32_t h0 = 0; h0 < nh; h0 += 64) {
			// the batch: lane t takes the region's (h0 + t)-th record
			const uint32_t cnt = min(64u, nh - h0);
			uint32_t np = 0;
			if (static_cast<uint32_t>(t) < cnt) {
				const IoRec r = rn;
				stri[t] = r;
				// its quads among the region's (both grids step 2 from even origins)
				const int minx = static_cast<int>(r.minxy & 0xffffu), miny = static_cast<int>(r.minxy >> 16);
				const int x0 = max(minx - rx0, 0) >> 1, y0 = max(miny - ry0, 0) >> 1;
				const int x1 = min((minx - rx0) / 2 + static_cast<int>((r.meta >> 16) & 0xffu), kRegionDim / 2);
				const int y1 = min((miny - ry0) / 2 + static_cast<int>(r.meta >> 24), kRegionDim / 2);
				np = static_cast<uint32_t>((x1 - x0) * (y1 - y0));
				srect[t] = static_cast<uint32_t>(x0) | (static_cast<uint32_t>(y0) << 4) | (static_cast<uint32_t>(x1 - x0) << 8); }
			if (h0 + 64 + static_cast<uint32_t>(t) < nh) rn = record(h0 + 64 + static_cast<uint32_t>(t));
			uint32_t pend = np;   // pairs up to and with this lane's triangle
			for (int o = 1; o < 64; o <<= 1) {
				const uint32_t v = __shfl_up(pend, o, 64);
				if (t >= o) pend += v; }
			const uint32_t total = __shfl(pend, 63, 64), pbeg = pend - np;
			qoff[t] = pbeg;
			uint32_t nwait = 0;   // listed fragments
			for (uint32_t w0 = 0; w0 < total; w0 += 64) {
				// the window's pairs name their triangles
				for (uint32_t p = max(pbeg, w0), pe = min(pend, w0 + 64u); p < pe; ++p) wtri[p - w0] = static_cast<uint8_t>(t);
				__syncthreads();
				// cover: lane t takes pair w0 + t
				uint32_t live = 0, entry = 0;
				if (w0 + static_cast<uint32_t>(t) < total) {
					const int j = wtri[t];
					const uint32_t k = w0 + static_cast<uint32_t>(t) - qoff[j], rc = srect[j], cx = rc >> 8;
					const uint32_t iy = (k * (cx == 3u ? 22u : 64u >> (cx >> 1))) >> 6;   // k / cx for k < 16, cx <= 4
					const uint32_t wx = (rc & 15u) + k - iy * cx, wy = ((rc >> 4) & 15u) + iy;
					entry = static_cast<uint32_t>(j) | (wx << 8) | (wy << 10);
					const int px = rx0 + 2 * static_cast<int>(wx), py = ry0 + 2 * static_cast<int>(wy);
					const IoRec r = stri[j];
					const int32_t dx31 = wsub(0, wadd(r.dx12, r.dx23)), dy31 = wsub(0, wadd(r.dy12, r.dy23));
					const int kx = (px - static_cast<int>(r.minxy & 0xffffu)) >> 1, ky = (py - static_cast<int>(r.minxy >> 16)) >> 1;
					// the quad's lanes (c, c+dy, c+dx, c+dx+dy), stepped as the
					// rasteriser loops step (rglv_triangle.hxx:253-304)
					const int32_t q1 = wadd(wadd(r.c1, wmul(kx, wmul(r.dy12, 2))), wmul(ky, wmul(r.dx12, 2)));
					const int32_t q2 = wadd(wadd(r.c2, wmul(kx, wmul(r.dy23, 2))), wmul(ky, wmul(r.dx23, 2)));
					const int32_t q3 = wadd(wadd(r.c3, wmul(kx, wmul(dy31, 2))), wmul(ky, wmul(dx31, 2)));
					const int32_t e1[4] = { q1, wadd(q1, r.dy12), wadd(q1, r.dx12), wadd(wadd(q1, r.dx12), r.dy12) };
					const int32_t e2[4] = { q2, wadd(q2, r.dy23), wadd(q2, r.dx23), wadd(wadd(q2, r.dx23), r.dy23) };
					const int32_t e3[4] = { q3, wadd(q3, dy31), wadd(q3, dx31), wadd(wadd(q3, dx31), dy31) };
#pragma unroll
					for (int i = 0; i < 4; ++i) live |= ((e1[i] | e2[i] | e3[i]) >= 0 ? 1u : 0u) << i;
					const DrawLite& dl = lite[r.meta & 0xffu];
					if (live && dl.scissorOn) {
						// the scissor flags of the rasteriser loops mask exactly
						// the lanes outside the clipped raster rect (tile origins
						// are even)
						const Rect S = draw_tile_rect(dl, (R.x0 / f.tileW), (R.y0 / f.tileH));
#pragma unroll
						for (int i = 0; i < 4; ++i) {
							const int sx = px + (i & 1), sy = py + (i >> 1);
							if (sx < S.x0 || sx >= S.x1 || sy < S.y0 || sy >= S.y1) live &= ~(1u << i); }}}
				const uint32_t nlive = static_cast<uint32_t>(__popc(live));
				frags += nlive;
				uint32_t fend = nlive;   // covered fragments up to and with this lane's pair
				for (int o = 1; o < 64; o <<= 1) {
					const uint32_t v = __shfl_up(fend, o, 64);
					if (t >= o) fend += v; }
				const uint32_t nf = __shfl(fend, 63, 64);
				uint32_t fat = nwait + fend - nlive;
#pragma unroll
				for (int i = 0; i < 4; ++i) if ((live >> i) & 1u) flist[fat++] = static_cast<uint16_t>(entry | (static_cast<uint32_t>(i) << 6));
				nwait += nf;
				__syncthreads();
				// shade and apply whole rounds; what is left waits for the next
				// window's fragments, or is the batch's last round
				uint32_t f0 = 0;
				for (; nwait - f0 >= 64; f0 += 64) round(f0, 64);
				if (w0 + 64 >= total) {
					if (nwait > f0) round(f0, nwait - f0);
					nwait = 0; }
				else if (f0 > 0) {
					nwait -= f0;
					const uint16_t en = flist[f0 + static_cast<uint32_t>(t)];
					__syncthreads();
					flist[t] = en; }}
			__syncthreads(); }}
	while (opi < ope) { apply_op(ops[opi]); ++opi; }
	// fragments that reached the depth test, one atomic per region
	for (int o = 32; o > 0; o >>= 1) frags += __shfl_xor(frags, o, 64);
	if (t == 0 && frags) atomicAdd(&a.ctr->slot[blockIdx.x % kCtrSlots].fragments, static_cast<unsigned long long>(frags)); }

}  // namespace rgl
