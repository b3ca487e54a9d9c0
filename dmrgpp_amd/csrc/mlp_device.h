// Device functions of the learned preconditioner's network (4 -> 64 -> 64 -> 1, tanh, FP32),
// shared by its inference, training and Davidson kernels: one wave evaluates 16 samples at a
// time on the matrix units.
//
// Lane l = 16 g + c holds, for sample c of the tile, the hidden units o = 16 b + 4 g + r (block
// b < 4, register r < 4): the layout of the MFMA result D[4 g + r][c]. The same registers are the
// right operand of the next layer as they stand, since a contraction may take its k in any order:
// lane group g supplies its own units on the right and W2[o][those units] on the left. So nothing
// goes through LDS between layers, and the whole W2 stays in registers.
//
// Inference multiplies layer 2 on bf16 MFMAs with every finite FP32 operand split into three bf16
// parts (8 + 8 + 8 bits: h = bf16(v), m = bf16(v - h), l = v - h - m) and the six products down to
// 2^-17 of the leading one kept (l l, l m and m l, below 2^-25, are dropped), accumulated in FP32:
// the error of a whole network is smaller than with FP32 sums in order (figures at the inference
// kernel). An infinite weight has no parts; see MlpWeightsInfinite. The reason is the issue port: on gfx950 an FP32 (or FP64) MFMA keeps the
// vector ALU from issuing for its whole duration (32 MFMAs and 128 FMAs, two waves per SIMD: 1.85
// and 1.04 ms alone, 2.65 ms together), a bf16 MFMA does not (1.83 and 1.04 ms alone, 1.85
// together), and the tanh work alone keeps the vector ALU busy.
#pragma once

#include "mlp.h"

#include <hip/hip_runtime.h>

namespace dmk {

typedef float  mlp_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 mlp_b8 __attribute__((ext_vector_type(8)));

constexpr int kMlpTile   = 16;             // samples per wave and pass
constexpr int kMlpBlocks = kMlpHidden / 16; // 16-unit blocks of a hidden layer

__device__ inline mlp_f4 mlp_mma(float a, float b, mlp_f4 c)
{
	return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ inline mlp_f4 mlp_mma(mlp_b8 a, mlp_b8 b, mlp_f4 c)
{
	return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Eight FP32 values as three bf16 parts each; the differences are exact.
struct MlpSplit {
	mlp_b8 h, m, l;
	__device__ inline void set(int i, float v)
	{
		h[i]          = __bf16(v);
		const float d = v - float(h[i]);
		m[i]          = __bf16(d);
		l[i]          = __bf16(d - float(m[i]));
	}
	// For any finite value: past the largest bf16 the rest goes to m and l.
	__device__ inline void set_any(int i, float v)
	{
		const float top = 3.3895314e38f;
		h[i]            = __bf16(v > top ? top : v < -top ? -top : v);
		const float d   = v - float(h[i]);
		m[i]            = __bf16(d);
		l[i]            = __bf16(d - float(m[i]));
	}
};

// tanh in FP32, odd: x + x^3 P(x^2) below 1 (P: minimax polynomial of (tanh(x)/x - 1)/x^2, fitted for
// this; 5e-9), 1 - 2 / (1 + exp(2 |x|)) with x's sign from the hardware exp2 and reciprocal above;
// +-1 at infinity, NaN for NaN. Both branches are computed, without divergence. Against 64 bits, over
// 8.4e6 arguments in [1e-8, 10] and their negatives: at most 1.22 units in the last place (7.3e-8),
// 0.277 rms; tanhf 1.34 (8.0e-8) and 0.279, in 1.2 times the time. The line lies at 1 because the
// exponential's error is larger just above it: at 0.8 the maximum is 1.40 (and 5 % less time), at 0.6
// 1.59 (9 % less).
__device__ inline float mlp_tanh(float x)
{
	const float ax = fabsf(x);
	const float t  = __builtin_amdgcn_exp2f(2.88539008f * ax);
	const float m  = __builtin_amdgcn_rcpf(1.0f + t);
	const float s  = x * x;
	float       p  = -3.58451944e-4f;
	p              = fmaf(p, s, 2.30136444e-3f);
	p              = fmaf(p, s, -7.94610567e-3f);
	p              = fmaf(p, s, 2.14866567e-2f);
	p              = fmaf(p, s, -5.38798012e-2f);
	p              = fmaf(p, s, 1.33323446e-1f);
	p              = fmaf(p, s, -3.33332956e-1f);
	const float lo = fmaf(x * s, p, x);
	const float hi = copysignf(fmaf(-2.0f, m, 1.0f), x);
	return ax < 1.0f ? lo : hi;
}

// The forward weights of one wave: left operands of both layers in registers; biases and W3
// (which only depend on the lane group) are read from the workgroup's LDS copy per tile.
struct MlpWeights {
	float    w1[kMlpBlocks];    // W1[16 b + c][g]
	MlpSplit w2[kMlpBlocks][2]; // [b2][s]: W2[16 b2 + c][k], k = 32 s + 16 (i / 4) + 4 g + i % 4

	__device__ inline void load(const float* __restrict__ params, int c, int g)
	{
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			w1[b] = params[kMlpOffW1 + (16 * b + c) * kMlpIn + g];
#pragma unroll
		for (int b2 = 0; b2 < kMlpBlocks; ++b2)
#pragma unroll
			for (int s = 0; s < 2; ++s)
#pragma unroll
				for (int i = 0; i < 8; ++i)
					w2[b2][s].set_any(i, params[kMlpOffW2 + (16 * b2 + c) * kMlpHidden + 32 * s
					                        + 16 * (i >> 2) + 4 * g + (i & 3)]);
	}
};

// The same where W2 holds an infinity, which has no parts (its products with the parts of a number
// would be NaN where one of those is 0): layer 2 on FP32 MFMAs, its rows from global memory.
struct MlpWeightsInfinite {
	float        w1[kMlpBlocks];
	const float* w2; // row c, from column 4 g on

	__device__ inline void load(const float* __restrict__ params, int c, int g)
	{
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			w1[b] = params[kMlpOffW1 + (16 * b + c) * kMlpIn + g];
		w2 = params + kMlpOffW2 + c * kMlpHidden + 4 * g;
	}
};

// Whether W2 holds an infinity; the same in every lane of the wave. The kernels ask before they
// load their weights and choose their loop by it: both forms in one loop do not fit three waves per
// SIMD, and 64 loads per lane, once per wave, are in flight together.
__device__ inline bool mlp_infinite(const float* __restrict__ params, int lane)
{
	bool inf = false;
#pragma unroll 16
	for (int i = 0; i < kMlpHidden * kMlpHidden / 64; ++i)
		inf |= isinf(params[kMlpOffW2 + 64 * i + lane]);
	return __ballot(inf) != 0;
}

// Biases of both layers and the output layer, in LDS.
struct MlpSmall {
	float b1[kMlpHidden], b2[kMlpHidden], w3[kMlpHidden];
	float b3;

	// By the first 64 threads of the workgroup; a barrier must follow.
	__device__ inline void load(const float* __restrict__ params, int tid)
	{
		if (tid < kMlpHidden) {
			b1[tid] = params[kMlpOffB1 + tid];
			b2[tid] = params[kMlpOffB2 + tid];
			w3[tid] = params[kMlpOffW3 + tid];
		}
		if (tid == 0)
			b3 = params[kMlpOffB3];
	}
	__device__ inline mlp_f4 at(const float* v, int b, int g) const
	{
		return *reinterpret_cast<const mlp_f4*>(v + 16 * b + 4 * g);
	}
};

// Keeps the compiler from holding the LDS biases in registers across tiles (48 registers: with
// W2's 64 they would leave three waves per SIMD, or spill).
__device__ inline void mlp_tile_fence() { asm volatile("" ::: "memory"); }

// h2 += W2 tanh(h1).
__device__ inline void mlp_layer2(const MlpWeights& w, const mlp_f4 h1[kMlpBlocks], mlp_f4 h2[kMlpBlocks])
{
#pragma unroll
	for (int s = 0; s < 2; ++s) {
		MlpSplit v;
#pragma unroll
		for (int i = 0; i < 8; ++i)
			v.set(i, mlp_tanh(h1[2 * s + (i >> 2)][i & 3]));
		// Small products first, and four independent accumulators between two uses of one.
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			h2[b] = mlp_mma(w.w2[b][s].l, v.h, h2[b]);
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			h2[b] = mlp_mma(w.w2[b][s].h, v.l, h2[b]);
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			h2[b] = mlp_mma(w.w2[b][s].m, v.m, h2[b]);
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			h2[b] = mlp_mma(w.w2[b][s].m, v.h, h2[b]);
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			h2[b] = mlp_mma(w.w2[b][s].h, v.m, h2[b]);
#pragma unroll
		for (int b = 0; b < kMlpBlocks; ++b)
			h2[b] = mlp_mma(w.w2[b][s].h, v.h, h2[b]);
	}
}

__device__ inline void mlp_layer2(const MlpWeightsInfinite& w, const mlp_f4 h1[kMlpBlocks],
                                  mlp_f4 h2[kMlpBlocks])
{
#pragma unroll
	for (int b = 0; b < kMlpBlocks; ++b)
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			const float v = mlp_tanh(h1[b][r]);
#pragma unroll
			for (int b2 = 0; b2 < kMlpBlocks; ++b2)
				h2[b2] = mlp_mma(w.w2[16 * b2 * kMlpHidden + 16 * b + r], v, h2[b2]);
			mlp_tile_fence(); // a few loads at a time
		}
}

// The network's output for sample c of a tile (in every lane group); x is feature g of sample c.
template <typename W>
__device__ inline float mlp_forward_tile(const W& w, const MlpSmall& sm, int g, float x)
{
	mlp_f4 h1[kMlpBlocks], h2[kMlpBlocks];
#pragma unroll
	for (int b = 0; b < kMlpBlocks; ++b) {
		h1[b] = mlp_mma(w.w1[b], x, sm.at(sm.b1, b, g));
		h2[b] = sm.at(sm.b2, b, g);
	}
	mlp_layer2(w, h1, h2);
	float y = 0.0f;
#pragma unroll
	for (int b = 0; b < kMlpBlocks; ++b) {
		const mlp_f4 w3 = sm.at(sm.w3, b, g);
#pragma unroll
		for (int r = 0; r < 4; ++r)
			y = fmaf(w3[r], mlp_tanh(h2[b][r]), y);
	}
	// The sum over the four lane groups, the same in each.
	y += __shfl_xor(y, 16);
	y += __shfl_xor(y, 32);
	return y + sm.b3;
}

} // namespace dmk
