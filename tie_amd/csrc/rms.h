// rms.h -- TIE's RMSNorm scale (rms_norm_f32_f32_f32_avx2, math_avx2.c:56-96,
// as TIE's build computes it) as device routines, shared by the RMSNorm
// kernel and the one-launch decode, which normalises its token itself.
#pragma once
#include "common.h"

namespace tie {

// the host's RSQRTSS of a positive normal float through the table
__device__ __forceinline__ float rsqrt_host(float a, const uint32_t *tab, int nbits)
{
	const uint32_t b = __builtin_bit_cast(uint32_t, a);
	const int eb = (int)(b >> 23);
	if (eb == 0)
		return __builtin_inff(); // zero (eps = 0 and an all-zero row)
	const int p = (eb - 126) & 1;
	const int s = (eb - 126 - p) >> 1;
	const uint32_t y = tab[(p << nbits) + ((b & 0x7fffffu) >> (23 - nbits))];
	return __builtin_bit_cast(float, y - (uint32_t)(s * (1 << 23)));
}

// the row's scale from its sum of squares ss (hsum8 of the eight chains)
__device__ __forceinline__ float rms_scale(float ss, int d, float eps, const uint32_t *tab, int nbits)
{
	const float a = __fdiv_rn(ss, (float)d) + eps;
	const float y0 = rsqrt_host(a, tab, nbits);
	return __builtin_fmaf(a * y0, y0, -3.0f) * (y0 * -0.5f);
}

} // namespace tie
