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
// times 1/16.
struct KawaseSrc {
	const float4* p;
	int W, H, stride;
	__device__ float4 at(int x, int y) const {
		x = x < 0 ? 0 : x > W - 1 ? W - 1 : x;
		y = y < 0 ? 0 : y > H - 1 ? H - 1 : y;
		return p[static_cast<long long>(y) * stride + x]; }
	// the box with its upper left texel at (x, y)
	__device__ float4 box(int x, int y) const {
		const float4 a = at(x, y), b = at(x + 1, y), c = at(x, y + 1), e = at(x + 1, y + 1);
		return make_float4(((a.x + b.x) + c.x) + e.x, ((a.y + b.y) + c.y) + e.y, ((a.z + b.z) + c.z) + e.z, ((a.w + b.w) + c.w) + e.w); }
};
__device__ inline float4 kawase_mean(const float4& b0, const float4& b1, const float4& b2, const float4& b3) {
	const float k16 = 1.0F / 16.0F;
	return make_float4(((((0.0F + b0.x) + b1.x) + b2.x) + b3.x) * k16, ((((0.0F + b0.y) + b1.y) + b2.y) + b3.y) * k16,
	                   ((((0.0F + b0.z) + b1.z) + b2.z) + b3.z) * k16, ((((0.0F + b0.w) + b1.w) + b2.w) + b3.w) * k16); }

// One thread per output pixel, 64 x 4 per workgroup so that a wave reads
// whole rows: sixteen texels a pixel through the vector cache.
__global__ __launch_bounds__(256) void k_kawase(const float4* __restrict__ src, float4* __restrict__ dst, int W, int H,
                                                int srcStride, int dstStride, int d) {
	const int x = static_cast<int>(blockIdx.x) * 64 + static_cast<int>(threadIdx.x & 63);
	const int y = static_cast<int>(blockIdx.y) * 4 + static_cast<int>(threadIdx.x >> 6);
	if (x >= W || y >= H) return;
	const KawaseSrc s{ src, W, H, srcStride };
	dst[static_cast<long long>(y) * dstStride + x] =
		kawase_mean(s.box(x - d - 1, y - d - 1), s.box(x + d, y - d - 1), s.box(x - d - 1, y + d), s.box(x + d, y + d)); }

// The same where four pixels share each box: a workgroup of 32 x 16 pixels
// keeps its (32 + 2d + 1) x (16 + 2d + 1) boxes in LDS, at d = 3 1.75 a pixel
// instead of four, so seven texels are read instead of sixteen.  What bounds
// k_kawase is the vector cache (16 bytes a lane take 16 clocks a wave).
// 1920 x 1080, us a pass, k_kawase and tiles: d = 0 19.1 and 14.2, 1 20.4 and
// 15.2, 3 20.1 and 17.0, 5 20.2 and 18.9, 7 18.1 and 20.8; at 960 x 540 and
// below both wait for the caller's launches (7).
constexpr int kKawaseX = 32, kKawaseY = 16;
constexpr int kKawaseMaxD = 5;   // 19 KB of boxes, 2.3 a pixel
constexpr int kawase_boxes(int d) { return (kKawaseX + 2 * d + 1) * (kKawaseY + 2 * d + 1); }

__global__ __launch_bounds__(256) void k_kawase_tile(const float4* __restrict__ src, float4* __restrict__ dst, int W, int H,
                                                     int srcStride, int dstStride, int d) {
	extern __shared__ float4 boxes[];   // kawase_boxes(d)
	const int t = static_cast<int>(threadIdx.x), reach = 2 * d + 1, bw = kKawaseX + reach, n = kawase_boxes(d);
	const int x0 = static_cast<int>(blockIdx.x) * kKawaseX, y0 = static_cast<int>(blockIdx.y) * kKawaseY;
	const KawaseSrc s{ src, W, H, srcStride };
	const float rbw = 1.0F / static_cast<float>(bw);
	for (int i = t; i < n; i += 256) {
		// i / bw: below 1,161, and (i + 0.5) / bw is off an integer by 0.5 / 43 at least
		const int by = static_cast<int>((static_cast<float>(i) + 0.5F) * rbw);
		boxes[i] = s.box(x0 - d - 1 + i - by * bw, y0 - d - 1 + by); }
	__syncthreads();
	const int x = x0 + (t & 31);
#pragma unroll
	for (int r = 0; r < 2; ++r) {
		const int y = y0 + (t >> 5) + 8 * r;
		const float4* q = boxes + ((t >> 5) + 8 * r) * bw + (t & 31);
		if (x < W && y < H)
			dst[static_cast<long long>(y) * dstStride + x] = kawase_mean(q[0], q[reach], q[reach * bw], q[reach * bw + reach]); }}

}  // namespace rgl
