// norm.hip -- the RMSNorm in front of the MoE block (model_qwen3.c:392-401).
//
// rms_norm_f32_f32_f32_avx2 (math_avx2.c:56-96) as TIE's build computes it:
//   ss  = hsum8 of eight FMA chains, chain l over x[8i + l] (i ascending)
//   a   = ss / size + eps                       (IEEE divide and add)
//   y0  = RSQRTSS(a)                            (the host CPU's approximation)
//   inv = fma(a * y0, y0, -3) * (y0 * -0.5)     (GCC's Newton step)
//   out = (x * w) * inv
// RSQRTSS comes from a table built on the host at set-up (its output depends
// only on the exponent parity and the top `nbits` mantissa bits; the
// exponent scales exactly), so the kernel reproduces TIE's bits.
#include "common.h"
#include "rms.h"
#include "route.h"

namespace tie {

// One wave (a workgroup of its own) per token.  The wave requests a chunk of
// the row at once, 16 bytes per lane and load, and stores it to LDS by chain:
// chain l's elements x[8i + l] are contiguous (row stride padded by 4 floats,
// so the 16-byte reads of lanes 0..7 fall in different banks); lanes 0..7
// then run the eight sum-of-squares chains four elements per LDS read.  Then
// the whole wave scales the row, from registers where one chunk holds it.
// Bound by latency: the launch, one memory round trip, TIE's chain of d / 8
// dependent FMAs (about 1 us at d = 2048), the table look-up.  Four tokens per
// workgroup with a load at a time took 9.8 us at T = 101, d = 2048 (now 4.7),
// 12.3 at T = 2000 (8.8), 18.2 at T = 300, d = 4096 (8.0).
constexpr int NORM_CHUNK = 2048;               // floats of a row staged at a time
constexpr int NORM_V = NORM_CHUNK / 256;       // float4 per lane and chunk
constexpr int NORM_LSTRIDE = NORM_CHUNK / 8 + 4; // floats per chain row in LDS
__global__ __launch_bounds__(64) void rmsnorm_kernel(const float *__restrict__ x, const float *__restrict__ w, float eps,
						     int d, float *__restrict__ out, const uint32_t *__restrict__ tab,
						     int nbits)
{
	__shared__ __attribute__((aligned(16))) float buf[8 * NORM_LSTRIDE];
	const int lane = threadIdx.x;
	const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)blockIdx.x * d);
	const float4 *wr = reinterpret_cast<const float4 *>(w);
	const int n4 = d / 4; // a multiple of 64
	float4 v[NORM_V], wv[NORM_V];
	float acc = 0.0f;
	for (int c0 = 0; c0 < n4; c0 += 64 * NORM_V) {
#pragma unroll
		for (int j = 0; j < NORM_V; j++)
			v[j] = xr[min(c0 + 64 * j, n4 - 64) + lane];
		if (n4 <= 64 * NORM_V)
#pragma unroll
			for (int j = 0; j < NORM_V; j++)
				wv[j] = wr[min(64 * j, n4 - 64) + lane];
#pragma unroll
		for (int j = 0; j < NORM_V; j++) {
			// float4 c of the chunk goes to chains 4 (c % 2) + 0..3, position c / 2
			const int c = 64 * j + lane;
			float *o = buf + 4 * (c & 1) * NORM_LSTRIDE + (c >> 1);
			o[0] = v[j].x;
			o[NORM_LSTRIDE] = v[j].y;
			o[2 * NORM_LSTRIDE] = v[j].z;
			o[3 * NORM_LSTRIDE] = v[j].w;
		}
		__syncthreads();
		const int n = min(NORM_CHUNK, d - 4 * c0); // a multiple of 256
		if (lane < 8) {
			const float *ch = buf + lane * NORM_LSTRIDE;
#pragma unroll 8
			for (int i = 0; i < n / 8; i += 4) {
				const float4 q = *reinterpret_cast<const float4 *>(ch + i);
				acc = __builtin_fmaf(q.x, q.x, acc);
				acc = __builtin_fmaf(q.y, q.y, acc);
				acc = __builtin_fmaf(q.z, q.z, acc);
				acc = __builtin_fmaf(q.w, q.w, acc);
			}
		}
		__syncthreads();
	}
	const float ss = hsum8_lanes(acc); // lane 0
	float inv = lane == 0 ? rms_scale(ss, d, eps, tab, nbits) : 0.0f;
	inv = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, inv)));
	float4 *o = reinterpret_cast<float4 *>(out + (size_t)blockIdx.x * d);
	auto scale = [&](const float4 &xv, const float4 &wv) {
		return make_float4((xv.x * wv.x) * inv, (xv.y * wv.y) * inv, (xv.z * wv.z) * inv, (xv.w * wv.w) * inv);
	};
	if (n4 <= 64 * NORM_V) {
#pragma unroll
		for (int j = 0; j < NORM_V; j++)
			if (64 * j < n4)
				o[64 * j + lane] = scale(v[j], wv[j]);
	} else {
#pragma unroll 4
		for (int c = lane; c < n4; c += 64)
			o[c] = scale(xr[c], wr[c]);
	}
}

hipError_t launch_rmsnorm(const float *x, const float *w, float eps, int T, int d, float *out, const uint32_t *tab,
			  int nbits, hipStream_t s)
{
	if (T == 0)
		return hipSuccess;
	tie_launch(rmsnorm_kernel, dim3(T), dim3(64), 0, s, x, w, eps, d, out, tab, nbits);
	return hipGetLastError();
}

} // namespace tie
