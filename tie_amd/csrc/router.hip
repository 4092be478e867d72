// router.hip -- router logits, top-k selection and softmax gate weights.
//
// Reference: dispatch_mat_vec on ffn_gate_inp (model_qwen3.c:431-432) runs
// mat_vec_row_f32_f32_f32_avx2 (math_avx2.c:228-256): per expert row, 8
// lane accumulators acc[l] += x[8i+l] * w[8i+l] (FMA, i ascending), then
// the hsum_f32_avx2 tree (math_avx2.c:14-21).  find_top_k (engine.c:891-914)
// and softmax over the k selected logits (engine.c:864-888) follow.  The
// kernels below keep those exact operation sequences, so logits, selected
// experts and gate weights are bit-identical to TIE's.
//
// Logit kernels (no cross-workgroup handshakes: an agent-scope fence costs
// more than a launch on this multi-XCD part):
//   router_small   T <= 4: one workgroup per expert row, row and tokens
//                  staged in LDS, one thread per (token, lane) chain.
//   router_mid     2 to 32 tokens, and any number where there is no copy of
//                  the matrix in router_mm's order (E not a multiple of 16;
//                  F32 matrices of tie_hip_mat_mat): one workgroup per
//                  (expert, 16 or 32 tokens), row in LDS, x streamed from L2.
//   router_mm      more: the chains on the fp32 matrix cores.
// Selection kernel: router_topk (a wave per token, E <= 1024).  Small
// batches select and group in one workgroup instead (route_group_kernel,
// dispatch.hip).
#include "common.h"
#include "route.h"

namespace tie {

// Words the next kernels accumulate into (the matrix-core path's per-expert
// pair counts and token masks, and its recomputation count), cleared by
// the logits kernel's workgroups (grid-strided)
__device__ __forceinline__ void zero_words(const ZeroArgs &z)
{
	const int nb = gridDim.x * gridDim.y, b = blockIdx.y * gridDim.x + blockIdx.x;
	for (int i = b * blockDim.x + threadIdx.x; i < z.n; i += nb * blockDim.x)
		z.p[i] = 0;
	for (int i = b * blockDim.x + threadIdx.x; i < z.n2; i += nb * blockDim.x)
		z.p2[i] = 0;
	if (z.one && b == 0 && threadIdx.x == 0)
		*z.one = 0;
}

// ------------------------------------------------------------ router_small
// One token (RS_TOK at most): one workgroup per expert row; the row and the tokens are
// staged in LDS with coalesced 16-byte loads and thread (t, l) runs the
// lane-l chain of token t.  Spreads the 1 MiB router matrix over E
// workgroups, which matters most at T = 1.
constexpr int RS_TOK = 4;
// router_small only for one token: from 2 tokens on router_mid is faster
// (T=4: 11 -> 8.2 us)
#ifndef TIE_RS_MAX_T
#define TIE_RS_MAX_T 1
#endif
constexpr int RS_THREADS = 256;

__global__ __launch_bounds__(RS_THREADS) void router_small_kernel(const float *__restrict__ x,
								  const float *__restrict__ W,
								  const float *__restrict__ bias, int T, int d, int E,
								  float *__restrict__ logits, ZeroArgs z)
{
	zero_words(z);
	extern __shared__ float lds[]; // W row | x [RS_TOK], lane-major (lane_chain)
	float *ws = lds;
	float *xs = lds + lane_major_floats(d);
	const int e = blockIdx.x;
	const int nt = min(RS_TOK, T);
	const int tid = threadIdx.x;

	// the row and the tokens -> LDS, lane-major
	stage_lane_major(ws, W + (size_t)e * d, d);
	for (int t = 0; t < nt; t++)
		stage_lane_major(xs + t * lane_major_floats(d), x + (size_t)t * d, d);
	__syncthreads();
	if (tid >= RS_TOK * 8)
		return;
	const int t = tid >> 3, l = tid & 7;
	const float acc = t < nt ? lane_chain(xs + (size_t)t * lane_major_floats(d), ws, d, l) : 0.0f;
	const float r = hsum8_lanes(acc);
	if (l == 0 && t < nt)
		logits[(size_t)t * E + e] = bias ? r + bias[e] : r;
}

// ------------------------------------------------------------ router_mid
// RS_TOK < T (up to a few hundred tokens): one workgroup per (expert, TOK
// tokens).  The expert row is staged in LDS (read as a broadcast); thread
// (t, l) streams x[t][8i + l] from global memory (L2-resident) with many
// loads in flight and runs the lane-l chain of token t.  TOK tokens per
// workgroup: 16 up to 32 tokens (twice the workgroups, over more CUs),
// else 32.
// U: inputs per lane and batch (d a multiple of 8 U).  LM: the row staged
// lane-major, its weights read a batch ahead in 16-byte reads (263
// registers: one wave per SIMD, so only while one round of workgroups
// covers the grid: up to 64 tokens)
template <int U, int TOK, bool LM>
__global__ __launch_bounds__(TOK * 8) void router_mid_kernel(const float *__restrict__ x,
							     const float *__restrict__ W,
							     const float *__restrict__ bias, int T, int d, int E,
							     float *__restrict__ logits, ZeroArgs z)
{
	zero_words(z);
	extern __shared__ float ws[]; // W row [d]
	const int e = blockIdx.x;
	constexpr int RM_THREADS = TOK * 8;
	const int t0 = blockIdx.y * TOK;
	const int tid = threadIdx.x;
	const int t = t0 + (tid >> 3), l = tid & 7;
	const bool live = t < T;
	const float *xt = x + (size_t)(live ? t : 0) * d + l;
	// the token's inputs stream in batches of U per lane, the next batch
	// loading while the current one is multiplied; the first batch is
	// issued before the row's staging, so the two memory waits overlap
	const int nbt = d / (8 * U);
	float xa[U], xb[U];
#pragma unroll
	for (int u = 0; u < U; u++)
		xa[u] = xt[8 * u];
	float acc = 0.0f;
	if constexpr (LM) {
		// the row lane-major (lane l's weights 8i + l contiguous): one 16-byte
		// LDS read brings 4 steps, and the next batch's weights are read while
		// the current batch is multiplied
		typedef float f4 __attribute__((ext_vector_type(4)));
		stage_lane_major(ws, W + (size_t)e * d, d);
		__syncthreads();
		const f4 *wl = reinterpret_cast<const f4 *>(ws + l * lane_major_stride(d));
		constexpr int U4 = U / 4;
		f4 wa[U4], wb[U4];
#pragma unroll
		for (int q = 0; q < U4; q++)
			wa[q] = wl[q];
		for (int bt = 0; bt < nbt; bt += 2) {
			if (bt + 1 < nbt) {
#pragma unroll
				for (int u = 0; u < U; u++)
					xb[u] = xt[8 * U * (bt + 1) + 8 * u];
#pragma unroll
				for (int q = 0; q < U4; q++)
					wb[q] = wl[U4 * (bt + 1) + q];
			}
#pragma unroll
			for (int u = 0; u < U; u++)
				acc = __builtin_fmaf(xa[u], wa[u / 4][u % 4], acc);
			if (bt + 1 >= nbt)
				break;
			if (bt + 2 < nbt) {
#pragma unroll
				for (int u = 0; u < U; u++)
					xa[u] = xt[8 * U * (bt + 2) + 8 * u];
#pragma unroll
				for (int q = 0; q < U4; q++)
					wa[q] = wl[U4 * (bt + 2) + q];
			}
#pragma unroll
			for (int u = 0; u < U; u++)
				acc = __builtin_fmaf(xb[u], wb[u / 4][u % 4], acc);
	}
	} else {
		const float4 *W4 = reinterpret_cast<const float4 *>(W + (size_t)e * d);
		for (int i = tid; i < (d >> 2); i += RM_THREADS)
			reinterpret_cast<float4 *>(ws)[i] = W4[i];
		__syncthreads();
		const float *wl = ws + l;
		for (int bt = 0; bt < nbt; bt += 2) {
			if (bt + 1 < nbt) {
#pragma unroll
				for (int u = 0; u < U; u++)
					xb[u] = xt[8 * U * (bt + 1) + 8 * u];
			}
#pragma unroll
			for (int u = 0; u < U; u++)
				acc = __builtin_fmaf(xa[u], wl[8 * U * bt + 8 * u], acc);
			if (bt + 1 >= nbt)
				break;
			if (bt + 2 < nbt) {
#pragma unroll
				for (int u = 0; u < U; u++)
					xa[u] = xt[8 * U * (bt + 2) + 8 * u];
			}
#pragma unroll
			for (int u = 0; u < U; u++)
				acc = __builtin_fmaf(xb[u], wl[8 * U * (bt + 1) + 8 * u], acc);
	}
	}
	const float r = hsum8_lanes(acc);
	if (l == 0 && live)
		logits[(size_t)t * E + e] = bias ? r + bias[e] : r;
}

// ------------------------------------------------------------ router_mm
// TIE's chains on the fp32 matrix cores.  v_mfma_f32_16x16x4_f32 computes
// D[m][n] = fma(a[m][3], b[3][n], fma(a[m][2], b[2][n], fma(a[m][1], b[1][n],
// fma(a[m][0], b[0][n], C[m][n])))) with every step rounded as v_fma_f32
// rounds it (compared bit for bit over ordinary values, denormals,
// infinities and NaN: 1.5 M results of each kind), so with K index kk =
// step 4s + kk of chain l it is exactly 4 steps of TIE's lane-l accumulator
// for 16 tokens x 16 experts, at twice the FMA rate of the vector unit and
// a 16th of its operand reads per FMA.
//
// One workgroup (8 waves) per 16 NT tokens x 16 NE experts; wave w runs chain
// l = w.  K advances RM_KC = 256 inputs (8 MFMAs per chain and 16 x 16 tile)
// at a time: the x rows come in by coalesced 16-byte loads RM_PD chunks ahead
// and are transposed through a double-buffered LDS tile to the operand order;
// the weights are stored in operand order at layer creation
// (launch_router_order) and go straight to registers, RM_PD chunks ahead too.
// Operand order, for chain l and 16 steps: lane (kk = lane / 16, r = lane %
// 16) holds steps 4c + kk, c = 0..3, of row r in one 16-byte word.
//
// Bound: the matrix pipe at large T (T d E FMAs at 32 per clock and SIMD: 6.8
// us at 2048 x 2048 x 128; the kernel without its loads and LDS traffic took
// 15 us there), else the latency of the launch and the first loads (about 4
// us) and of the chunks.  Against the kernels it replaced (LDS-tiled vector
// FMAs above 256 tokens, router_mid below; 30B shape, same card): T=64 7.7 ->
// 6.9 us, T=101 11.5 -> 7.3, T=256 19.7 -> 7.0, T=500 17.9 -> 9.3, T=1024
// 19.4 -> 12.5, T=2048 28.2 -> 19.4; 235B T=1024 35.0 -> 19.6.  Up to 32
// tokens router_mid stays: T=32 6.3 us against 7.2, T=8 5.0 against 6.5.
// Four waves of two chains each, and 3, 4 or 6 chunks ahead: within 3%.
constexpr int RM_NW = 8, RM_PD = 2, RM_MIN_T = 32;
constexpr int RM_KC = 256, RM_G = RM_KC / 128;
// LDS strides of the x tile (floats): K group of 4 lanes' rows, 16-step
// group, chain; the writes of a wave (32 steps of 2 chains) then fall in
// distinct banks, two lanes a bank
constexpr int RM_SK = 68, RM_SG = 4 * RM_SK, RM_SL = RM_G * RM_SG + 8, RM_BUF = 8 * RM_SL;

typedef float rm_f4 __attribute__((ext_vector_type(4)));

// whether 4 consecutive x values leave the f16 range (XConvArgs)
__device__ __forceinline__ int rm_bad(const float4 a)
{
	const float m = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(a.x), __builtin_fabsf(a.y)),
					__builtin_fmaxf(__builtin_fabsf(a.z), __builtin_fabsf(a.w)));
	// fmax drops NaN: test the values themselves for NaN
	const bool nan = a.x != a.x || a.y != a.y || a.z != a.z || a.w != a.w;
	return (nan || !(m < 65504.0f)) ? 1 : 0;
}

template <int NE, int NT, bool CONV>
__global__ __launch_bounds__(64 * RM_NW) __attribute__((amdgpu_waves_per_eu(2))) void
router_mm_kernel(const float *__restrict__ x, const float *__restrict__ WM, const float *__restrict__ bias, int T, int d,
		 int E, float *__restrict__ logits, int by_token, ZeroArgs z, XConvArgs xc)
{
	constexpr int NW = RM_NW, PD = RM_PD;
	constexpr int TOK = 16 * NT;       // tokens per workgroup
	constexpr int XR = TOK / NW;       // x rows per wave
	constexpr int BUF = NT * RM_BUF;   // floats of one half of the x tile
	zero_words(z);
	__shared__ __attribute__((aligned(16))) float xs[2 * BUF];
	const int tid = threadIdx.x, lane = tid & 63;
	const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
	// workgroups go round-robin over the 8 XCDs, each with its own L2:
	// consecutive ids take different token tiles with the expert tiles of a
	// token tile on one XCD (by_token: x is the larger operand), or
	// different expert tiles
	const int net = E / (16 * NE), ntt = (T + TOK - 1) / TOK;
	int tt, et;
	if (by_token) {
		tt = (int)(blockIdx.y * 8 + blockIdx.x % 8);
		et = (int)blockIdx.x / 8;
		if (tt >= ntt)
			return;
	} else {
		et = (int)blockIdx.x % net;
		tt = (int)blockIdx.x / net;
	}
	const int t0 = tt * TOK, nt = min(TOK, T - t0);
	const int nck = d / RM_KC;

	// x: thread loads float4 c4 = lane of rows w + NW j (rows past the batch
	// re-read the last one: their outputs are not stored), at 32-bit offsets
	// from a wave-uniform base
	const char *xbase = reinterpret_cast<const char *>(x + (size_t)t0 * d);
	uint32_t xo[XR];
#pragma unroll
	for (int j = 0; j < XR; j++)
		xo[j] = (uint32_t)(min(w + NW * j, nt - 1) * d * 4 + lane * 16);
	// its place in the tile: chains 4 (lane % 2) + 0..3, step i = lane / 2
	const int st = lane >> 1;
	float *xw = xs + 4 * (lane & 1) * RM_SL + (st >> 4) * RM_SG + (st & 3) * RM_SK + ((st >> 2) & 3);
	// weights: tile et, chain l, step group g: 64 lanes x 16 bytes
	const uint32_t tile = (uint32_t)d * 64; // bytes of a tile (16 experts)
	const char *wbase = reinterpret_cast<const char *>(WM) + (size_t)et * NE * tile + (size_t)w * (tile / 8);
	const uint32_t wo = lane * 16;

	float4 xv[PD][XR];
	rm_f4 wv[PD][NE][RM_G];
	auto load_x = [&](int ck, float4 (&v)[XR]) {
		const char *b = xbase + min(ck, nck - 1) * (RM_KC * 4);
#pragma unroll
		for (int j = 0; j < XR; j++)
			v[j] = *reinterpret_cast<const float4 *>(b + xo[j]);
	};
	auto load_w = [&](int ck, rm_f4 (&v)[NE][RM_G]) {
		const char *b = wbase + min(ck, nck - 1) * (RM_G * 1024);
#pragma unroll
		for (int n = 0; n < NE; n++)
#pragma unroll
			for (int g = 0; g < RM_G; g++)
				v[n][g] = *reinterpret_cast<const rm_f4 *>(b + n * tile + g * 1024 + wo);
	};
#pragma unroll
	for (int p = 0; p < PD; p++) {
		load_x(p, xv[p]);
		load_w(p, wv[p]);
	}
	rm_f4 acc[NT][NE];
#pragma unroll
	for (int m = 0; m < NT; m++)
#pragma unroll
		for (int n = 0; n < NE; n++)
			acc[m][n] = rm_f4{0.0f, 0.0f, 0.0f, 0.0f};
	int bad[XR] = {};

	const int kk = lane >> 4, r = lane & 15;
	const float *rb = xs + w * RM_SL + kk * RM_SK + 4 * r;
	rm_f4 a[NT][RM_G];
	// element c of x row j out of its register into chunk ck's half of the tile
	auto put = [&](int ck, int j, int c, const float4 &v) {
		const int row = w + NW * j;
		xw[(ck & 1) * BUF + (row >> 4) * RM_BUF + 4 * (row & 15) + c * RM_SL] = c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
	};
	// a share of the chunks per expert tile goes to the f16 A operand too
	auto convert = [&](int ck, const float4 (&v)[XR]) {
#pragma unroll
		for (int j = 0; j < XR; j++) {
			typedef _Float16 h4 __attribute__((ext_vector_type(4)));
			const int row = w + NW * j;
			bad[j] |= rm_bad(v[j]);
			if (row < nt)
				*reinterpret_cast<h4 *>(xc.xa + (size_t)(t0 + row) * d + ck * RM_KC + 4 * lane) =
					h4{(_Float16)v[j].x, (_Float16)v[j].z, (_Float16)v[j].y, (_Float16)v[j].w};
		}
	};
	auto get = [&](int ck) {
#pragma unroll
		for (int m = 0; m < NT; m++)
#pragma unroll
			for (int g = 0; g < RM_G; g++)
				a[m][g] = *reinterpret_cast<const rm_f4 *>(rb + (ck & 1) * BUF + m * RM_BUF + g * RM_SG);
	};
#pragma unroll
	for (int j = 0; j < XR; j++)
#pragma unroll
		for (int c = 0; c < 4; c++)
			put(0, j, c, xv[0][j]);
	if (CONV && et == 0)
		convert(0, xv[0]);
	load_x(PD, xv[0]);
	__syncthreads();
	get(0);
	// chunk ck (weights in slot p; p a constant after unrolling): its MFMAs,
	// with the next chunk's writes to the other half of the tile and, into the
	// freed registers, the loads of chunks ck + 1 + PD (x) and ck + PD
	// (weights) issued one after each MFMA, under its 32 cycles.  The fences
	// keep that order.
	auto step = [&](int ck, int p, bool more) {
		constexpr int M = 8 * NT * NE, W = 4 * XR;
		const int pn = (p + 1) % PD;
		if (CONV && (ck + 1) % net == et && ck + 1 < nck)
			convert(ck + 1, xv[pn]);
		const char *bx = xbase + min(ck + 1 + PD, nck - 1) * (RM_KC * 4);
		const char *bw = wbase + min(ck + PD, nck - 1) * (RM_G * 1024) + wo;
#pragma unroll
		for (int u = 0; u < M; u++) {
			const int n = u % NE, m = u / NE % NT, q = u / (NE * NT) % 4, g = u / (M / RM_G);
			acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][g][q], wv[p][n][g][q], acc[m][n], 0, 0, 0);
#pragma unroll
			for (int i = u * W / M; i < (u + 1) * W / M; i++) {
				// (past the last chunk: a copy nothing reads)
				put(ck + 1, i / 4, i % 4, xv[pn][i / 4]);
				if (more && i % 4 == 3)
					xv[pn][i / 4] = *reinterpret_cast<const float4 *>(bx + xo[i / 4]);
			}
			__builtin_amdgcn_sched_barrier(0);
			if (more && (u + 1) % (M / RM_G) == 0) {
				// a step group's weights are used up
#pragma unroll
				for (int i = 0; i < NE; i++)
					wv[p][i][g] = *reinterpret_cast<const rm_f4 *>(bw + i * tile + g * 1024);
				__builtin_amdgcn_sched_barrier(0);
			}
		}
		__syncthreads();
		get(ck + 1);
	};
	int c0 = 0;
	for (; c0 + PD <= nck; c0 += PD)
#pragma unroll
		for (int p = 0; p < PD; p++)
			step(c0 + p, p, true);
#pragma unroll
	for (int p = 0; p < PD - 1; p++)
		if (c0 + p < nck)
			step(c0 + p, p, false);
	if (CONV) {
		// this expert tile's share of a token's flag: the OR over its wave's
		// lanes (the routing kernel ORs the tiles')
#pragma unroll
		for (int j = 0; j < XR; j++) {
			const int any = __any(bad[j]);
			if (lane == 0 && w + NW * j < nt)
				xc.part[(size_t)(t0 + w + NW * j) * net + et] = any ? 1 : 0;
		}
	}
	// hsum8: s_m = v[m] + v[m + 4], (s0 + s1) + (s2 + s3) (math_avx2.c:14-21
	// order), over the waves through LDS.  D layout: lane l, register i:
	// token 4 (l / 16) + i, expert l % 16.
	constexpr int OT = 16 * 17; // floats of one wave's 16 x 16 sums
	static_assert(NT * NE * NW * OT <= 2 * BUF, "sums in the x tile");
	__syncthreads();
#pragma unroll
	for (int m = 0; m < NT; m++)
#pragma unroll
		for (int n = 0; n < NE; n++)
#pragma unroll
			for (int i = 0; i < 4; i++)
				xs[((m * NE + n) * NW + w) * OT + (4 * kk + i) * 17 + r] = acc[m][n][i];
	__syncthreads();
	for (int o = tid; o < TOK * 16 * NE; o += 64 * NW) {
		const int c = o % (16 * NE), t = o / (16 * NE);
		const float *q = xs + (((t >> 4) * NE + (c >> 4)) * NW) * OT + (t & 15) * 17 + (c & 15);
		float s4[4];
#pragma unroll
		for (int m = 0; m < 4; m++)
			s4[m] = q[m * OT] + q[(m + 4) * OT];
		const float sum = (s4[0] + s4[1]) + (s4[2] + s4[3]);
		const int e = et * 16 * NE + c;
		if (t < nt)
			logits[(size_t)(t0 + t) * E + e] = bias ? sum + bias[e] : sum;
	}
}

// W [E][d] -> the operand order of router_mm_kernel (once, at layer
// creation; E a multiple of 16): [E / 16][chain 8][d / 128][lane 64][4]
__global__ void router_order_kernel(const float *__restrict__ W, float *__restrict__ WM, int E, int d)
{
	const size_t n = (size_t)E * d, step = (size_t)gridDim.x * blockDim.x;
	const int ng = d / 128;
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
		const int q = (int)(i & 3), lane = (int)(i >> 2) & 63;
		const size_t u = i >> 8;
		const int g = (int)(u % ng), l = (int)(u / ng) & 7, et = (int)(u / ng / 8);
		WM[i] = W[(size_t)(16 * et + (lane & 15)) * d + 8 * (16 * g + 4 * q + (lane >> 4)) + l];
	}
}

hipError_t launch_router_order(const Layer &L, hipStream_t s)
{
	if (L.E % 16)
		return hipSuccess; // no operand order: the row kernels serve every T
	tie_launch(router_order_kernel, dim3(256), dim3(256), 0, s, L.router, (float *)L.routerM, L.E, L.d);
	return hipGetLastError();
}

// ------------------------------------------------------------ router_topk
// one wave per token (topk_softmax, E <= MAX_E)
constexpr int RW_THREADS = 256;
__global__ __launch_bounds__(RW_THREADS) void router_topk_kernel(const float *__restrict__ logits, int T, int E,
								      int k, int32_t *__restrict__ topk_idx,
								      float *__restrict__ topk_w, int routing,
								      const float *__restrict__ pbias)
{
	__shared__ uint64_t etab[32];
	if (threadIdx.x < 32) {
		const uint64_t tab[32] = TIE_EXP2_TABLE;
		etab[threadIdx.x] = tab[threadIdx.x];
	}
	__syncthreads();
	const int t = blockIdx.x * (RW_THREADS / 64) + (threadIdx.x >> 6);
	if (t < T)
		topk_softmax(logits + (size_t)t * E, E, k, etab, topk_idx + (size_t)t * k, topk_w + (size_t)t * k, routing,
			     pbias);
}

static bool router_on_mm(const Layer &L, int T)
{
	return T > RM_MIN_T && L.E % 16 == 0 && L.routerM;
}

bool router_converts_x(const Layer &L, int T)
{
	// (up to 256 tokens the routing kernel, a wave per token, converts the rows
	// under its selection; above, sharing it with the logits is faster: 30B
	// T=2048 19.4 + 7.0 us against 17.1 + 10.4)
	return T > 256 && router_on_mm(L, T);
}

hipError_t launch_router_logits(const Layer &L, const float *x, int T, float *logits, hipStream_t s, ZeroArgs z,
				XConvArgs *conv)
{
	const int d = L.d, E = L.E;
	if (T <= TIE_RS_MAX_T && sizeof(float) * (size_t)(8 * (d / 8 + 4)) * (1 + RS_TOK) <= 160 * 1024) {
		const size_t lds = sizeof(float) * (size_t)(8 * (d / 8 + 4)) * (1 + RS_TOK);
		tie_launch(router_small_kernel, dim3(E), dim3(RS_THREADS), lds, s, x, L.router, L.bias, T, d, E,
				   logits, z);
		return hipGetLastError();
	}
	if (router_on_mm(L, T)) {
		auto go = [&](auto kern, int tok, int exp) {
			const int ntt = (T + tok - 1) / tok, net = E / exp;
			const int by_token = T >= 256 ? 1 : 0; // x the larger operand
			if (conv)
				conv->tiles = net;
			// 8 token tiles x all expert tiles in x, groups of 8 in y (at most a
			// 128th of the tokens: the combine has a token in each y)
			tie_launch(kern, by_token ? dim3(8 * net, (ntt + 7) / 8) : dim3(ntt * net), dim3(64 * RM_NW), 0, s, x,
				   L.routerM, L.bias, T, d, E, logits, by_token, z, conv ? *conv : XConvArgs());
		};
		// larger tiles (fewer x transpositions and weight reads per MFMA) once
		// they still cover most of the CUs: 30B T=500 (64 tiles of 32 x 32)
		// 9.3 us with 16 x 16 tiles, 12.5 with 16 x 32, 16.9 with 32 x 32;
		// T=1024 (128) 16.6 / 12.5 / 17.5; T=1500 (188) 18.8 with 16 x 32, 18.5
		// with 32 x 32; T=2048 (256) 23.6 / 19.4
		const int t32 = E % 32 == 0 ? (T + 31) / 32 * (E / 32) : 0;
		if (t32 >= 192)
			conv ? go(router_mm_kernel<2, 2, true>, 32, 32) : go(router_mm_kernel<2, 2, false>, 32, 32);
		else if (t32 >= 96)
			conv ? go(router_mm_kernel<2, 1, true>, 16, 32) : go(router_mm_kernel<2, 1, false>, 16, 32);
		else
			conv ? go(router_mm_kernel<1, 1, true>, 16, 16) : go(router_mm_kernel<1, 1, false>, 16, 16);
		return hipGetLastError();
	}
	const bool u64 = d % 512 == 0;
	const int tok = T <= 32 ? 16 : 32;
	const bool lm = T <= 64;
	auto kern = lm ? (tok == 16 ? (u64 ? router_mid_kernel<64, 16, true> : router_mid_kernel<32, 16, true>)
				    : (u64 ? router_mid_kernel<64, 32, true> : router_mid_kernel<32, 32, true>))
		       : (u64 ? router_mid_kernel<64, 32, false> : router_mid_kernel<32, 32, false>);
	tie_launch(kern, dim3(E, (T + tok - 1) / tok), dim3(tok * 8),
			   sizeof(float) * (size_t)(lm ? lane_major_floats(d) : d), s, x, L.router, L.bias, T, d, E, logits, z);
	return hipGetLastError();
}

hipError_t launch_router_select(const Layer &L, int T, int k, const float *logits, int32_t *topk_idx, float *topk_w,
				hipStream_t s)
{
	tie_launch(router_topk_kernel, dim3((T + RW_THREADS / 64 - 1) / (RW_THREADS / 64)), dim3(RW_THREADS), 0,
			   s, logits, T, L.E, k, topk_idx, topk_w, L.routing, L.pbias);
	return hipGetLastError();
}

hipError_t launch_router(const Layer &L, const float *x, int T, int k, float *logits, int32_t *topk_idx,
			 float *topk_w, hipStream_t s)
{
	hipError_t err = launch_router_logits(L, x, T, logits, s);
	if (err != hipSuccess)
		return err;
	return launch_router_select(L, T, k, logits, topk_idx, topk_w, s);
}

} // namespace tie
