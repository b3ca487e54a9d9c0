// The learned Davidson preconditioner: a per-element MLP (4 -> 64 -> 64 -> 1, tanh), FP32,
// with its inference, gradient and optimizer kernels.
//
// Parameters are one flat FP32 array: W1 (64 x 4, row major: W1[o][i]), b1 (64), W2 (64 x 64,
// W2[o][i]), b2 (64), W3 (64), b3 (1). A forward pass per element x (4 features):
//   h1 = tanh(W1 x + b1), h2 = tanh(W2 h1 + b2), y = W3 . h2 + b3.
// The gradient of the mean squared error over a batch is accumulated per workgroup in a fixed
// sample order and the workgroup partials are summed in index order, so a gradient is bitwise
// reproducible.
#include "dmk_internal.h"
#include "mlp.h"
#include "mlp_device.h"

#include <hip/hip_runtime.h>

namespace dmk {

namespace {

constexpr int kT      = 256; // threads per workgroup
constexpr int kPass   = 64;  // samples per pass of the gradient kernel
constexpr int kLd     = kMlpHidden + 4; // LDS row: 16-byte aligned, 4 banks further per row

} // namespace

// y[s] = MLP(x[s]) for count samples (features row major, kMlpIn per sample): each wave takes
// tiles of 16 samples, grid-stride, the next tile's features loaded during the current one.
// Bound by the vector ALU: 128 tanh per sample and the splits of layer 1's results, about 740
// vector and 64 transcendental operations per tile (0.25 ms for 2.86e6 samples); the bf16 MFMAs
// (52 per tile) run beside them, with three waves per SIMD. 2.86e6 samples, whole call: 4.97 ms
// with one sample per thread (weights in LDS, activations in scratch), 0.29 ms now (0.27 with a
// tanh of 3.7 units in the last place); error of y against 64 bits, five networks of a trained
// one's size on features N(0, 1): 1.7e-7 to 3.7e-7 with one sample per thread, 1.1e-7 to 2.7e-7 now.
__global__ __launch_bounds__(kT) __attribute__((amdgpu_waves_per_eu(3))) void mlp_forward_kernel(
    const float* __restrict__ params, const float* __restrict__ x, int64_t count,
    float* __restrict__ y)
{
	__shared__ __attribute__((aligned(16))) MlpSmall sm;
	sm.load(params, threadIdx.x);
	const int  lane = threadIdx.x & 63;
	const int  c = lane & 15, g = lane >> 4;
	const bool infinite = mlp_infinite(params, lane);
	__syncthreads();
	const int64_t step = int64_t(gridDim.x) * (kT / 64) * kMlpTile;
	const int64_t first = (int64_t(blockIdx.x) * (kT / 64) + (threadIdx.x >> 6)) * kMlpTile;
	if (first >= count)
		return;
	auto feature = [&](int64_t t0) {
                const int64_t s = t0 + c < count ? t0 + c : count - 1; // past the end: unused
                return x[s * kMlpIn + g];
	};
	auto run = [&](auto w) {
		float xn = feature(first);
		w.load(params, c, g);
		for (int64_t s0 = first; s0 < count; s0 += step) {
			mlp_tile_fence();
			const float xi = xn;
			if (s0 + step < count)
				xn = feature(s0 + step);
			const float out = mlp_forward_tile(w, sm, g, xi);
			if (g == 0 && s0 + c < count)
				y[s0 + c] = out;
		}
	};
	if (infinite)
		run(MlpWeightsInfinite {});
	else
		run(MlpWeights {});
}

// Per-workgroup partial gradient of L = (1/N) sum_s (y_s - t_s)^2 over samples
// [0, count) of (x, t), N = count: partial[wg * (kMlpParams + 1) + p], the last entry holding
// the partial sum of squared errors (LOSS: that entry alone). Workgroup wg takes passes of kPass
// samples wg, wg + G, ... in order; each of its four waves carries 16 of a pass's samples through
// both layers and back in the register layout of mlp_device.h, where the transposed contraction
// (W2^T times the deltas) also needs no exchange. The weight gradients contract over the samples,
// so activations and deltas go through LDS once, unit by unit, and wave w then owns the rows
// 16 w .. 16 w + 15 of every gradient, in accumulators that live across the passes. The right
// operand of the small gradients holds the features, 1 and dL/dy as columns: one MFMA each gives
// (W1, b1), b2 and W3.
//
// FP32 MFMAs throughout (sums in FP32 as before). A batch is a few microseconds of latency (one
// pass per workgroup and CU at most): 64 samples per pass and one workgroup per CU spread it over
// as many CUs as it has passes. 8192 samples: 106 us with the layers on the vector ALU out of LDS,
// 11.7 us now, of which 3.3 us are MFMAs; the loss alone over 262144 samples 43 us.
template <bool LOSS>
__global__ __launch_bounds__(kT) __attribute__((amdgpu_waves_per_eu(1))) void mlp_grad_kernel(
    const float* __restrict__ params, const float* __restrict__ x, const float* __restrict__ t,
    int64_t count, float* __restrict__ partial)
{
	constexpr int NB = kMlpBlocks;
	__shared__ __attribute__((aligned(16))) MlpSmall sm;
	__shared__ __attribute__((aligned(16))) float    W2[kMlpHidden][kLd];
	// [unit][sample of the pass]
	__shared__ __attribute__((aligned(16))) float H1[LOSS ? 1 : kMlpHidden][kLd];
	__shared__ __attribute__((aligned(16))) float H2[LOSS ? 1 : kMlpHidden][kLd];
	__shared__ __attribute__((aligned(16))) float DA1[LOSS ? 1 : kMlpHidden][kLd];
	__shared__ __attribute__((aligned(16))) float DA2[LOSS ? 1 : kMlpHidden][kLd];
	__shared__ float X[kPass][kMlpIn];
	__shared__ float DY[kPass];
	__shared__ float red[2][kT / 64];
	const int tid  = threadIdx.x;
	const int lane = tid & 63, wave = tid >> 6;
	const int c = lane & 15, g = lane >> 4;
	auto      vec4 = [](const float* p) { return *reinterpret_cast<const mlp_f4*>(p); };
	// The lane's sample of a pass; loaded a pass ahead, the first beside the weights.
	const int ls   = kMlpTile * wave + c;
	float     xn   = 0.0f, tn = 0.0f;
	auto      next = [&](int64_t pass) {
                const int64_t s = pass * kPass + ls;
                xn              = s < count ? x[s * kMlpIn + g] : 0.0f;
                tn              = s < count ? t[s] : 0.0f;
	};
	next(blockIdx.x);
	sm.load(params, tid);
#pragma unroll
	for (int q = 0; q < kMlpHidden * kMlpHidden / kT; ++q) {
		const int e                           = tid + kT * q;
		W2[e / kMlpHidden][e % kMlpHidden] = params[kMlpOffW2 + e];
	}
	float w1[NB];
#pragma unroll
	for (int b = 0; b < NB; ++b)
		w1[b] = params[kMlpOffW1 + (16 * b + c) * kMlpIn + g];
	__syncthreads();
	mlp_f4 w2[NB][NB];  // [b2][b]: W2[16 b2 + c][16 b + 4 g ..]
	mlp_f4 w2t[NB][NB]; // [b][b2]: W2[16 b2 + 4 g + r][16 b + c]
#pragma unroll
	for (int b2 = 0; b2 < NB; ++b2)
#pragma unroll
		for (int b = 0; b < NB; ++b) {
			w2[b2][b] = vec4(&W2[16 * b2 + c][16 * b + 4 * g]);
			if constexpr (!LOSS)
#pragma unroll
				for (int r = 0; r < 4; ++r)
					w2t[b][b2][r] = W2[16 * b2 + 4 * g + r][16 * b + c];
		}
	const float   scale = 2.0f / float(count);
	const int64_t npass = (count + kPass - 1) / kPass;
	mlp_f4        gw2[NB], gx = {}, gb2 = {}, gw3 = {};
#pragma unroll
	for (int b = 0; b < NB; ++b)
		gw2[b] = mlp_f4 {};
	float accse = 0.0f, accdy = 0.0f;
	for (int64_t pass = blockIdx.x; pass < npass; pass += gridDim.x) {
		const bool  valid = pass * kPass + ls < count;
		const float xi = xn, ti = tn;
		if (pass + gridDim.x < npass)
			next(pass + gridDim.x);
		// Forward.
		mlp_f4 h1[NB], h2[NB];
#pragma unroll
		for (int b = 0; b < NB; ++b) {
			h1[b] = mlp_mma(w1[b], xi, sm.at(sm.b1, b, g));
			h2[b] = sm.at(sm.b2, b, g);
#pragma unroll
			for (int r = 0; r < 4; ++r)
				h1[b][r] = mlp_tanh(h1[b][r]);
		}
#pragma unroll
		for (int b = 0; b < NB; ++b)
#pragma unroll
			for (int r = 0; r < 4; ++r)
#pragma unroll
				for (int b2 = 0; b2 < NB; ++b2)
					h2[b2] = mlp_mma(w2[b2][b][r], h1[b][r], h2[b2]);
		float y = 0.0f;
#pragma unroll
		for (int b = 0; b < NB; ++b) {
			const mlp_f4 w3 = sm.at(sm.w3, b, g);
#pragma unroll
			for (int r = 0; r < 4; ++r) {
				h2[b][r] = mlp_tanh(h2[b][r]);
				y        = fmaf(w3[r], h2[b][r], y);
			}
		}
		y += __shfl_xor(y, 16);
		y += __shfl_xor(y, 32);
		const float err = valid ? y + sm.b3 - ti : 0.0f;
		accse           = fmaf(err, err, accse);
		if constexpr (!LOSS) {
			// Back: da2 = dL/d(pre-activation 2), da1 likewise.
			const float dy = scale * err;
			accdy += dy;
			mlp_f4 da2[NB], da1[NB];
#pragma unroll
			for (int b = 0; b < NB; ++b) {
				const mlp_f4 w3 = sm.at(sm.w3, b, g);
				da1[b]          = mlp_f4 {};
#pragma unroll
				for (int r = 0; r < 4; ++r)
					da2[b][r] = dy * w3[r] * (1.0f - h2[b][r] * h2[b][r]);
			}
#pragma unroll
			for (int b2 = 0; b2 < NB; ++b2)
#pragma unroll
				for (int r = 0; r < 4; ++r)
#pragma unroll
					for (int b = 0; b < NB; ++b)
						da1[b] = mlp_mma(w2t[b][b2][r], da2[b2][r], da1[b]);
			__syncthreads(); // the previous pass's contractions have read the arrays
#pragma unroll
			for (int b = 0; b < NB; ++b)
#pragma unroll
				for (int r = 0; r < 4; ++r) {
					const int o = 16 * b + 4 * g + r;
					H1[o][ls]   = h1[b][r];
					H2[o][ls]   = h2[b][r];
					DA2[o][ls]  = da2[b][r];
					DA1[o][ls]  = da1[b][r] * (1.0f - h1[b][r] * h1[b][r]);
				}
			X[ls][g] = xi;
			if (g == 0)
				DY[ls] = dy;
			__syncthreads();
			// Over the pass's samples, 16 at a time: samples 16 q + 4 g + j for lane group g.
#pragma unroll 1
			for (int q = 0; q < kPass / 16; ++q) {
				const int    s4 = 16 * q + 4 * g;
				const mlp_f4 a2 = vec4(&DA2[16 * wave + c][s4]);
				const mlp_f4 a1 = vec4(&DA1[16 * wave + c][s4]);
				const mlp_f4 ah = vec4(&H2[16 * wave + c][s4]);
#pragma unroll
				for (int b = 0; b < NB; ++b) {
					const mlp_f4 hb = vec4(&H1[16 * b + c][s4]);
#pragma unroll
					for (int j = 0; j < 4; ++j)
						gw2[b] = mlp_mma(a2[j], hb[j], gw2[b]);
				}
#pragma unroll
				for (int j = 0; j < 4; ++j) {
					const float xv  = X[s4 + j][c & 3];
					const float dv  = DY[s4 + j];
					const float col = c < kMlpIn ? xv : c == 4 ? 1.0f : c == 5 ? dv : 0.0f;
					gx              = mlp_mma(a1[j], col, gx);
					gb2             = mlp_mma(a2[j], col, gb2);
					gw3             = mlp_mma(ah[j], col, gw3);
				}
			}
		}
	}
	// Sums over samples of the squared errors and of dL/dy, in a fixed order (each lane group of a
	// wave holds the same 16 values).
#pragma unroll
	for (int off = 1; off < 16; off <<= 1) {
		accse += __shfl_xor(accse, off);
		accdy += __shfl_xor(accdy, off);
	}
	if (lane == 0) {
		red[0][wave] = accse;
		red[1][wave] = accdy;
	}
	__syncthreads();
	float* out = partial + int64_t(blockIdx.x) * (kMlpParams + 1);
	if (tid == 0) {
		out[kMlpParams] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
		if (!LOSS)
			out[kMlpOffB3] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
	}
	if constexpr (!LOSS) {
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			const int o = 16 * wave + 4 * g + r;
#pragma unroll
			for (int b = 0; b < NB; ++b)
				out[kMlpOffW2 + o * kMlpHidden + 16 * b + c] = gw2[b][r];
			if (c < kMlpIn)
				out[kMlpOffW1 + o * kMlpIn + c] = gx[r];
			if (c == 4) {
				out[kMlpOffB1 + o] = gx[r];
				out[kMlpOffB2 + o] = gb2[r];
			}
			if (c == 5)
				out[kMlpOffW3 + o] = gw3[r];
		}
	}
}

// Arguments of the Adam step that the reduction applies (params null: none).
struct AdamStep {
	float* params;
	float* m;
	float* v;
	float  lr, b1, b2, eps;
	int    step;
};

// grad[p] = sum over workgroups of the partials for p0 <= p <= kMlpParams, and the Adam step
// (bias-corrected, step number `step` >= 1) on the parameters. 64 entries per workgroup, 16 waves
// that each sum every 16th partial in index order; the 16 sums are then added in order. The
// partials (2.3 MB for 128 workgroups) come from other XCDs' L2: all of a thread's loads are in
// flight together (one thread per entry, one load at a time, took 31 us, and the optimizer's own
// launch another 5; this takes 4.1 us).
constexpr int kRedWaves = 16;
__global__ __launch_bounds__(64 * kRedWaves) void mlp_reduce_kernel(
    const float* __restrict__ partial, int nparts, float* __restrict__ grad, int p0, AdamStep a)
{
	__shared__ float sum[kRedWaves][64];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int p = p0 + int(blockIdx.x) * 64 + lane;
	float     s = 0.0f;
	if (p <= kMlpParams) {
		float v[256 / kRedWaves];
#pragma unroll
		for (int q = 0; q < 256 / kRedWaves; ++q) {
			const int w = wave + kRedWaves * q;
			v[q]        = w < nparts ? partial[int64_t(w) * (kMlpParams + 1) + p] : 0.0f;
		}
#pragma unroll
		for (int q = 0; q < 256 / kRedWaves; ++q)
			s += v[q];
	}
	sum[wave][lane] = s;
	__syncthreads();
	if (wave != 0 || p > kMlpParams)
		return;
	float g = sum[0][lane];
#pragma unroll
	for (int w = 1; w < kRedWaves; ++w)
		g += sum[w][lane];
	grad[p] = g;
	if (a.params && p < kMlpParams) {
		const float c1 = 1.0f - powf(a.b1, float(a.step));
		const float c2 = 1.0f - powf(a.b2, float(a.step));
		const float mm = a.b1 * a.m[p] + (1.0f - a.b1) * g;
		const float vv = a.b2 * a.v[p] + (1.0f - a.b2) * g * g;
		a.m[p]         = mm;
		a.v[p]         = vv;
		a.params[p] -= a.lr * (mm / c1) / (sqrtf(vv / c2) + a.eps);
	}
}

int mlp_grad_parts(int64_t count)
{
	int64_t passes = (count + kPass - 1) / kPass;
	return int(passes < 256 ? (passes < 1 ? 1 : passes) : 256);
}

void launch_mlp_forward(const float* params, const float* x, int64_t count, float* y, hipStream_t s)
{
	if (count <= 0)
		return;
	// One tile per wave up to the 768 workgroups that are resident at once (three per CU); the
	// weights are loaded once per wave, so more workgroups only repeat that.
	int64_t b = (count + kMlpTile * (kT / 64) - 1) / (kMlpTile * (kT / 64));
	if (b > 768)
		b = 768;
	hipLaunchKernelGGL(mlp_forward_kernel, dim3(unsigned(b)), dim3(kT), 0, s, params, x, count, y);
	DMK_HIP_CHECK(hipGetLastError());
}

namespace {
void launch_reduce(const float* partial, int parts, float* grad, int p0, const AdamStep& a,
                   hipStream_t s)
{
	hipLaunchKernelGGL(mlp_reduce_kernel, dim3(unsigned((kMlpParams + 1 - p0 + 63) / 64)),
	                   dim3(64 * kRedWaves), 0, s, partial, parts, grad, p0, a);
	DMK_HIP_CHECK(hipGetLastError());
}
} // namespace

void launch_mlp_grad(const float* params, const float* x, const float* t, int64_t count,
                     float* partial, float* grad, hipStream_t s)
{
	const int parts = mlp_grad_parts(count);
	hipLaunchKernelGGL(mlp_grad_kernel<false>, dim3(unsigned(parts)), dim3(kT), 0, s, params, x, t,
	                   count, partial);
	DMK_HIP_CHECK(hipGetLastError());
	launch_reduce(partial, parts, grad, 0, AdamStep {}, s);
}

void launch_mlp_train_step(float* params, const float* x, const float* t, int64_t count,
                           float* partial, float* grad, float* m, float* v, float lr, int step,
                           hipStream_t s)
{
	const int parts = mlp_grad_parts(count);
	hipLaunchKernelGGL(mlp_grad_kernel<false>, dim3(unsigned(parts)), dim3(kT), 0, s, params, x, t,
	                   count, partial);
	DMK_HIP_CHECK(hipGetLastError());
	launch_reduce(partial, parts, grad, 0,
	              AdamStep { params, m, v, lr, 0.9f, 0.999f, 1e-8f, step }, s);
}

void launch_mlp_loss(const float* params, const float* x, const float* t, int64_t count,
                     float* partial, float* grad, hipStream_t s)
{
	const int parts = mlp_grad_parts(count);
	hipLaunchKernelGGL(mlp_grad_kernel<true>, dim3(unsigned(parts)), dim3(kT), 0, s, params, x, t,
	                   count, partial);
	DMK_HIP_CHECK(hipGetLastError());
	launch_reduce(partial, parts, grad, kMlpParams, AdamStep {}, s);
}

} // namespace dmk
