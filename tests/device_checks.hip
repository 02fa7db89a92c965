// Exhaustive checks of the scalar device functions whose bits every frame
// depends on, for all 2^32 inputs on the device.  Built beside the tests with
// the library's flags (rsr_amd.build.build_checks), called by
// test_device_functions_gpu.py.
#include <hip/hip_runtime.h>

#include "../rsr_amd/csrc/rgl_device.h"

namespace {

// f and its plain statement on one input's bits
enum Which { kRecip = 0, kRecipSqrt = 1, kRcpps = 2, kDepthOrder = 3, kCount = 4 };

// rcpps by its definition: a table entry, exponent 253 - e, zeros and
// subnormals to infinity, what leaves the exponents' range to zero
__device__ uint32_t rcpps_plain(uint32_t in) {
	const uint32_t e = (in >> 23) & 0xffu, s = in & 0x80000000u, m = in & 0x7fffffu;
	if (e == 0xffu) return m ? (in | 0x400000u) : s;
	if (e == 0u) return s | 0x7f800000u;
	const int re = 253 - static_cast<int>(e);
	return re <= 0 ? s : (s | (static_cast<uint32_t>(re) << 23) | rgl::kRcpMantissa[m >> 12]); }

__device__ uint32_t depth_order_plain(uint32_t u) {
	if (u == 0x80000000u) u = 0u;
	return (u & 0x80000000u) ? ~u : (u | 0x80000000u); }

__device__ bool differs(int which, uint32_t u) {
	const float x = rgl::u2f(u);
	switch (which) {
	case kRecip: return rgl::f2u(rgl::recip(x)) != rgl::f2u(1.0F / x);
	case kRecipSqrt: return rgl::f2u(rgl::recip_sqrt(x)) != rgl::f2u(1.0F / __builtin_sqrtf(x));
	case kRcpps: return rgl::f2u(rgl::rcpps(x)) != rcpps_plain(u);
	default: return x == x && rgl::depth_order(x) != depth_order_plain(u); }}   // NaN depths take no key

// out[0]: inputs that differ, out[1]: one of them
__global__ __launch_bounds__(256) void k_all(int which, unsigned long long* out) {
	const uint32_t first = (blockIdx.x * 256u + threadIdx.x) * 256u;   // 65,536 workgroups: all 2^32
	unsigned bad = 0;
	uint32_t one = 0;
	for (uint32_t k = 0; k < 256u; ++k)
		if (differs(which, first + k)) { ++bad; one = first + k; }
	if (bad) { atomicAdd(&out[0], static_cast<unsigned long long>(bad)); atomicMax(&out[1], static_cast<unsigned long long>(one)); }}

}  // namespace

extern "C" int rgl_check_all(int which, unsigned long long out[2]) {
	if (which < 0 || which >= kCount) return -1;
	unsigned long long* d = nullptr;
	if (hipMalloc(reinterpret_cast<void**>(&d), 16) != hipSuccess) return -2;
	const unsigned long long zero[2] = { 0, 0 };
	int r = hipMemcpy(d, zero, 16, hipMemcpyHostToDevice) == hipSuccess ? 0 : -2;
	if (r == 0) {
		hipLaunchKernelGGL(k_all, dim3(65536), dim3(256), 0, nullptr, which, d);
		if (hipGetLastError() != hipSuccess || hipMemcpy(out, d, 16, hipMemcpyDeviceToHost) != hipSuccess) r = -2; }
	(void)hipFree(d);
	return r; }
