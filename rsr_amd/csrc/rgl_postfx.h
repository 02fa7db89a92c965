// rgl_postfx.h — the float-canvas post effect of the rgl pipeline on
// gfx950: the Kawase blur pass (rglr_kawase.cxx:21-85).
#pragma once

#include "rgl_device.h"

namespace rgl {

// One Kawase pass over a W x H RGBA float canvas (row strides in pixels):
// each output pixel is the mean of four 2 x 2 boxes whose corners sit
// (d + 1) pixels up-left, up-right, down-left and down-right of it, with
// coordinates clamped to the canvas (KawaseBlurFilter's sample_safe; its
// unclamped interior loop reads the same texels).  Sums in the reference's
// order: the box ((a + b) + c) + d, the boxes accumulated from zero, then
// times 1/16.  One thread per output pixel, 64 x 4 per workgroup so that a
// wave reads whole rows.
__global__ __launch_bounds__(256) void k_kawase(const float4* __restrict__ src, float4* __restrict__ dst, int W, int H,
                                                int srcStride, int dstStride, int d) {
	const int x = static_cast<int>(blockIdx.x) * 64 + static_cast<int>(threadIdx.x & 63);
	const int y = static_cast<int>(blockIdx.y) * 4 + static_cast<int>(threadIdx.x >> 6);
	if (x >= W || y >= H) return;
	auto at = [&](int px, int py) {
		px = px < 0 ? 0 : px > W - 1 ? W - 1 : px;
		py = py < 0 ? 0 : py > H - 1 ? H - 1 : py;
		return src[static_cast<long long>(py) * srcStride + px]; };
	const int ox[4] = { -d - 1, d, -d - 1, d }, oy[4] = { -d - 1, -d - 1, d, d };
	float4 ax = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		const float4 a = at(x + ox[k], y + oy[k]), b = at(x + ox[k] + 1, y + oy[k]);
		const float4 c = at(x + ox[k], y + oy[k] + 1), e = at(x + ox[k] + 1, y + oy[k] + 1);
		ax.x = ax.x + (((a.x + b.x) + c.x) + e.x);
		ax.y = ax.y + (((a.y + b.y) + c.y) + e.y);
		ax.z = ax.z + (((a.z + b.z) + c.z) + e.z);
		ax.w = ax.w + (((a.w + b.w) + c.w) + e.w); }
	const float k16 = 1.0F / 16.0F;
	dst[static_cast<long long>(y) * dstStride + x] = make_float4(ax.x * k16, ax.y * k16, ax.z * k16, ax.w * k16); }

// The same pass for small d: a 2 x 2 box is a corner of four output pixels,
// so a workgroup sums the boxes of a 32 x 16 tile and its border of d + 1
// once (four taps each, through the cache) into LDS, and an output pixel
// reads its four.  Per output 4.4 taps (d = 0) to 7 (d = 3) and four LDS reads
// in place of 16 taps, of which 133 MB a pass went through the L1s of a
// 960 x 540 canvas.  From kKawaseMaxD on the border's boxes outnumber what is
// shared.
constexpr int kKawaseW = 32, kKawaseH = 16, kKawaseMaxD = 7;

__global__ __launch_bounds__(256) void k_kawase_boxes(const float4* __restrict__ src, float4* __restrict__ dst, int W, int H,
                                                      int srcStride, int dstStride, int d) {
	extern __shared__ float4 box[];   // box (i, j): the pixels (x0 + i, y0 + j) .. + 1
	const int bw = kKawaseW + 2 * d + 1, bh = kKawaseH + 2 * d + 1;
	const int tx = static_cast<int>(blockIdx.x) * kKawaseW, ty = static_cast<int>(blockIdx.y) * kKawaseH;
	const int x0 = tx - d - 1, y0 = ty - d - 1;
	const int lane = static_cast<int>(threadIdx.x & 31), row = static_cast<int>(threadIdx.x >> 5);
	for (int j = row; j < bh; j += 8) {
		const int ya = min(max(y0 + j, 0), H - 1), yb = min(max(y0 + j + 1, 0), H - 1);
		const float4* ra = src + static_cast<long long>(ya) * srcStride;
		const float4* rb = src + static_cast<long long>(yb) * srcStride;
		for (int i = lane; i < bw; i += 32) {
			const int xa = min(max(x0 + i, 0), W - 1), xb = min(max(x0 + i + 1, 0), W - 1);
			const float4 a = ra[xa], b = ra[xb], c = rb[xa], e = rb[xb];
			box[j * bw + i] = make_float4(((a.x + b.x) + c.x) + e.x, ((a.y + b.y) + c.y) + e.y,
			                              ((a.z + b.z) + c.z) + e.z, ((a.w + b.w) + c.w) + e.w); }}
	__syncthreads();
	const int x = tx + lane, s = 2 * d + 1;
	if (x >= W) return;
	const float k16 = 1.0F / 16.0F;
#pragma unroll
	for (int r = 0; r < kKawaseH / 8; ++r) {
		const int j = row + 8 * r, y = ty + j;
		if (y >= H) return;
		const float4* p = box + j * bw + lane;
		const float4* q = p + s * bw;
		const float4 a = p[0], b = p[s], c = q[0], e = q[s];
		dst[static_cast<long long>(y) * dstStride + x] = make_float4(
			((((0.0F + a.x) + b.x) + c.x) + e.x) * k16, ((((0.0F + a.y) + b.y) + c.y) + e.y) * k16,
			((((0.0F + a.z) + b.z) + c.z) + e.z) * k16, ((((0.0F + a.w) + b.w) + c.w) + e.w) * k16); }}

}  // namespace rgl
