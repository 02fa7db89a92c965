// rgl_assets.h — texture preparation of the asset path on gfx950: decoded
// RGBA8 images to float texels (rglr_texture_load.cxx:39-66), the
// power-of-two resample (rglr_texture.cxx:13-31) and the mip chain
// (rglr_texture.cxx:34-81).
#pragma once

#include "rgl_device.h"

namespace rgl {

// ryg::srgb8_to_float's 256 values (ryg-srgb.h:33-56), made once on the host
struct Srgb8Table { float v[256]; };

// PNGToTexture's texel loop: R, G, B through the sRGB table, A = a / 255,
// RGB times A when premultiplying.  One thread per texel.
__global__ __launch_bounds__(256) void k_texture_from_rgba8(const uchar4* __restrict__ src, float4* __restrict__ dst,
                                                             long long n, int premultiply, Srgb8Table tab) {
	const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= n) return;
	const uchar4 p = src[i];
	float4 o = make_float4(tab.v[p.x], tab.v[p.y], tab.v[p.z], static_cast<float>(p.w) / 255.0F);
	if (premultiply) { o.x = o.x * o.w; o.y = o.y * o.w; o.z = o.z * o.w; }
	dst[i] = o; }

// ensurePowerOf2: a dim x dim nearest resample of a w x h texture, source
// row / column int(i / (dim - 1) * (size - 1)) in double precision.
__global__ __launch_bounds__(256) void k_texture_pow2(const float4* __restrict__ src, int w, int h, float4* __restrict__ dst,
                                                       int dim) {
	const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= static_cast<long long>(dim) * dim) return;
	const int iy = static_cast<int>(i / dim), ix = static_cast<int>(i - static_cast<long long>(iy) * dim);
	const int sy = static_cast<int>(static_cast<double>(iy) / static_cast<double>(dim - 1) * static_cast<double>(h - 1));
	const int sx = static_cast<int>(static_cast<double>(ix) / static_cast<double>(dim - 1) * static_cast<double>(w - 1));
	dst[i] = src[static_cast<long long>(sy) * w + sx]; }

// one level of Texture::maybe_make_mipmap: texel (x, y) of the level of
// size `size` (rows from `dstRow`) is the 2 x 2 mean of the level above
// (rows from `srcRow`), summed ((a + b) + c) + d and divided by 4; rows of
// `stride` texels
__global__ __launch_bounds__(256) void k_mip_level(float4* __restrict__ buf, int stride, int srcRow, int dstRow, int size) {
	const int i = static_cast<int>(blockIdx.x) * blockDim.x + static_cast<int>(threadIdx.x);
	if (i >= size * size) return;
	const int y = i / size, x = i - y * size;
	const float4* r1 = buf + static_cast<long long>(srcRow + 2 * y) * stride + 2 * x;
	const float4* r2 = r1 + stride;
	const float4 a = r1[0], b = r1[1], c = r2[0], d = r2[1];
	buf[static_cast<long long>(dstRow + y) * stride + x] = make_float4(
		(((a.x + b.x) + c.x) + d.x) / 4.0F, (((a.y + b.y) + c.y) + d.y) / 4.0F,
		(((a.z + b.z) + c.z) + d.z) / 4.0F, (((a.w + b.w) + c.w) + d.w) / 4.0F); }

// The three steps above in one pass over a dim x dim texture (mip: with its
// chain below it, and zeros beside the chain): a workgroup takes 64 x 64
// texels, a wave 16 rows of them, a lane a column.  The base texels are
// decoded (and resampled) from the image, stored, and reduced in registers:
// a 2 x 2 mean takes two rows of a lane and the lane 2^l to the right, so a
// wave leaves levels 1 to 4 and the workgroup, through LDS, levels 5 and 6.
// k_mip_tail makes the levels above.  Every store of a row is contiguous.
// Bound: the 32 B written per texel.  A 1000 x 777 image takes 12 us; as 14
// launches (decode, resample, zero fill, copy, one per level) it took 53 us.
constexpr int kTexTile = 64;

// first row of mip level l >= 1 of a dim x dim texture
__device__ inline int mip_row(int dim, int l) { return 2 * dim - (dim >> (l - 1)); }

__device__ inline float4 shfl_down4(const float4& v, int d) {
	return make_float4(__shfl_down(v.x, d, 64), __shfl_down(v.y, d, 64), __shfl_down(v.z, d, 64), __shfl_down(v.w, d, 64)); }

// ((a + b) + c) + d over 4 (an exact scaling)
__device__ inline float4 mean4(const float4& a, const float4& b, const float4& c, const float4& d) {
	return make_float4((((a.x + b.x) + c.x) + d.x) * 0.25F, (((a.y + b.y) + c.y) + d.y) * 0.25F,
	                   (((a.z + b.z) + c.z) + d.z) * 0.25F, (((a.w + b.w) + c.w) + d.w) * 0.25F); }

__global__ __launch_bounds__(256) void k_texture_prepare(const uchar4* __restrict__ src, int w, int h, int premultiply,
		float4* __restrict__ dst, int dim, int mip, Srgb8Table tab) {
	__shared__ float stab[256];
	__shared__ int srow[kTexTile];
	__shared__ float4 sl4[4][4];
	stab[threadIdx.x] = tab.v[threadIdx.x];
	const int lane = static_cast<int>(threadIdx.x & 63), wv = static_cast<int>(threadIdx.x >> 6);
	const int bx = static_cast<int>(blockIdx.x) * kTexTile, by = static_cast<int>(blockIdx.y) * kTexTile;
	const bool resample = w != dim || h != dim;
	// source row / column int(i / (dim - 1) * (size - 1)) in double precision
	auto source = [&](int i, int size) {
		return resample ? static_cast<int>(static_cast<double>(i) / static_cast<double>(dim - 1) * static_cast<double>(size - 1)) : i; };
	if (wv == 0) srow[lane] = source(by + lane < dim ? by + lane : dim - 1, h);
	const int x = bx + lane, y0 = by + 16 * wv;
	const int sx = source(x < dim ? x : dim - 1, w);
	__syncthreads();
	const bool in = x < dim;
	uchar4 p[16];
#pragma unroll
	for (int k = 0; k < 16; ++k) p[k] = src[static_cast<long long>(srow[16 * wv + k]) * w + sx];
	float4 v[16];
#pragma unroll
	for (int k = 0; k < 16; ++k) {
		float4 o = make_float4(stab[p[k].x], stab[p[k].y], stab[p[k].z], static_cast<float>(p[k].w) / 255.0F);
		if (premultiply) { o.x = o.x * o.w; o.y = o.y * o.w; o.z = o.z * o.w; }
		v[k] = o;
		if (in && y0 + k < dim) dst[static_cast<long long>(y0 + k) * dim + x] = o; }
	if (!mip) return;
	// zeros beside the chain: row dim + y holds level l's texels, l the last
	// whose first row is at or before it, in its first dim >> l columns
#pragma unroll
	for (int k = 0; k < 16; ++k) {
		const int y = y0 + k;
		if (!in || y >= dim) continue;
		const int left = dim - 1 - y;                          // rows below this one
		const int width = left == 0 ? 0 : 1 << (31 - __clz(left));
		if (x >= width) dst[static_cast<long long>(dim + y) * dim + x] = make_float4(0.0F, 0.0F, 0.0F, 0.0F); }
#pragma unroll
	for (int l = 1; l <= 4; ++l) {
		const int size = dim >> l;   // texels across
#pragma unroll
		for (int k = 0; k < (16 >> l); ++k) {
			const float4 b = shfl_down4(v[2 * k], 1 << (l - 1)), d = shfl_down4(v[2 * k + 1], 1 << (l - 1));
			v[k] = mean4(v[2 * k], b, v[2 * k + 1], d);
			const int xl = x >> l, yl = (y0 >> l) + k;
			if ((lane & ((1 << l) - 1)) == 0 && xl < size && yl < size)
				dst[static_cast<long long>(mip_row(dim, l) + yl) * dim + xl] = v[k]; }}
	if (dim < 32) return;   // uniform: the chain has ended
	if ((lane & 15) == 0) sl4[wv][lane >> 4] = v[0];
	__syncthreads();
	if (threadIdx.x < 4) {
		const int i = static_cast<int>(threadIdx.x & 1), j = static_cast<int>(threadIdx.x >> 1);
		const float4 o = mean4(sl4[2 * j][2 * i], sl4[2 * j][2 * i + 1], sl4[2 * j + 1][2 * i], sl4[2 * j + 1][2 * i + 1]);
		const int xl = (bx >> 5) + i, yl = (by >> 5) + j;
		if (xl < (dim >> 5) && yl < (dim >> 5)) dst[static_cast<long long>(mip_row(dim, 5) + yl) * dim + xl] = o;
		const float4 b = shfl_down4(o, 1), c = shfl_down4(o, 2), d = shfl_down4(o, 3);
		if (threadIdx.x == 0 && dim >= 64)
			dst[static_cast<long long>(mip_row(dim, 6) + (by >> 6)) * dim + (bx >> 6)] = mean4(o, b, c, d); }}

// the levels above 6 of a texture of more than 64 texels (at most 4096): one
// workgroup, level 6's at most 64 x 64 texels in LDS
__global__ __launch_bounds__(1024) void k_mip_tail(float4* __restrict__ dst, int dim) {
	__shared__ float4 s[2][kTexTile * kTexTile];
	int size = dim >> 6, cur = 0;
	for (int i = static_cast<int>(threadIdx.x); i < size * size; i += 1024)
		s[0][i] = dst[static_cast<long long>(mip_row(dim, 6) + i / size) * dim + i % size];
	__syncthreads();
	for (int l = 7; size > 1; ++l, cur ^= 1) {
		const int half = size >> 1;
		for (int i = static_cast<int>(threadIdx.x); i < half * half; i += 1024) {
			const int y = i / half, x = i - y * half;
			const float4* r = s[cur] + 2 * y * size + 2 * x;
			const float4 o = mean4(r[0], r[1], r[size], r[size + 1]);
			s[cur ^ 1][i] = o;
			dst[static_cast<long long>(mip_row(dim, l) + y) * dim + x] = o; }
		__syncthreads();
		size = half; }}

}  // namespace rgl
