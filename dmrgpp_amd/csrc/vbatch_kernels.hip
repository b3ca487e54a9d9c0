// The variable-size batched GEMM kernel (dmk_gemm_vbatch_{d,z}): FP64 MFMA tiles straight from
// the caller's matrices into the caller's C.
//
// A workgroup (four waves, 2 x 2) owns a T x T tile of one product and walks k in chunks of 16
// elements. It computes the transposed product, C^T = op(B)^T op(A)^T, so that consecutive lanes
// of a result hold consecutive rows of the column-major C. Each operand is read along its own
// contiguous direction (along k where its columns run along k, else along its rows), 8 bytes (16
// complex) per lane with any alignment and leading dimension, through registers into LDS in that
// same orientation; the MFMA fragments are read from either layout. So transposes need no pass of
// their own, conjugation is a sign at the LDS store, and alpha and beta are applied in the result
// store. Rows past the edge repeat the last one, elements past k are zeroed in the last chunk.
//
// Loads are kept four chunks ahead in registers: a tile of a middle-sized block has few chunks
// and little company on its CU. Bound by the LDS (96 of 128 bytes per clock with 32 x 32 tiles) and,
// with 64 x 64 tiles, by the last round of tiles. On the wave-function transformation of an m = 2048
// ladder step (25 chains, 2.3 GFLOP per call) a launch takes 65 us, a call 93; staging the
// operands K-major in a workspace, the panel kernel and a scatter took 37 + 67 + 15 us, a call 224.
#include "dmk_internal.h"
#include "vbatch.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace dmk {

namespace {

constexpr int kVbThreads = 256;
constexpr int kVbK       = 16; // chunk of k
constexpr int kVbAhead   = 4;  // chunks in flight in registers (even: the LDS buffer of a step is static)

typedef double vd2 __attribute__((ext_vector_type(2)));
typedef double vd4 __attribute__((ext_vector_type(4)));
// A complex scalar at the caller's address (8-byte aligned).
typedef double vd2u __attribute__((ext_vector_type(2), aligned(8)));

// The caller's matrices as global memory: pointers read from a descriptor would be flat ones,
// whose loads also count as LDS operations and would be waited for at every barrier.
typedef const __attribute__((address_space(1))) char* vb_gptr;

// One operand tile: T rows (of op(A)^T or op(B)^T) x kVbK, one plane (real) or two (complex).
// ALONG_K: the source runs along k, LDS holds rows of 16-byte slots, XOR-swizzled as in the panel
// kernels; else the source runs along the rows, LDS holds k rows of T elements, padded so that
// k rows 4 apart (the lane groups of a fragment read) start 128 bytes apart modulo 256.
template <int T, bool ALONG_K, bool CPLX, bool WIDE> struct VbOperand {
	static constexpr int E   = T * kVbK / kVbThreads; // elements per thread and chunk
	static constexpr int LDK = T + 4;
	static constexpr int LDS = ALONG_K ? T * kVbK : kVbK * LDK; // doubles per plane
	using off_t              = typename std::conditional<WIDE, int64_t, uint32_t>::type;

	vb_gptr       base; // the tile's first row (wave-uniform)
	int64_t       step; // bytes per chunk of k
	off_t         off[E];
	int           kk[E];
	int64_t       ld;
	double        sign;

	__device__ inline static int krow(int e) { return ALONG_K ? e % kVbK : e / T; }
	__device__ inline static int trow(int e) { return ALONG_K ? e / kVbK : e % T; }

	__device__ inline void setup(const double* p, int ldp, int row0, int nrows, bool conj, int tid)
	{
		constexpr int C = CPLX ? 2 : 1;
		ld              = ldp;
		base            = (vb_gptr)(p + (ALONG_K ? int64_t(row0) * ld : int64_t(row0)) * C);
		step            = (ALONG_K ? int64_t(kVbK) : int64_t(kVbK) * ld) * C * int64_t(sizeof(double));
		sign            = conj ? -1.0 : 1.0;
#pragma unroll
		for (int q = 0; q < E; ++q) {
			const int e = tid + kVbThreads * q;
			const int r = min(row0 + trow(e), nrows - 1) - row0;
			kk[q]       = krow(e);
			off[q]      = offset(r, kk[q]);
		}
	}
	__device__ inline off_t offset(int r, int k) const
	{
		constexpr int C = CPLX ? 2 : 1;
		return off_t((ALONG_K ? off_t(r) * off_t(ld) + off_t(k) : off_t(k) * off_t(ld) + off_t(r))
		             * off_t(C * sizeof(double)));
	}
	// Whole chunk c into registers.
	__device__ inline void load(int c, vd2 v[E]) const
	{
		const vb_gptr p = base + c * step;
#pragma unroll
		for (int q = 0; q < E; ++q)
			v[q] = read(p + off[q]);
	}
	// The last `left` < kVbK elements, from chunk c, and zeros.
	__device__ inline void load_tail(int c, int left, vd2 v[E]) const
	{
		const vb_gptr p = base + c * step;
#pragma unroll
		for (int q = 0; q < E; ++q) {
			const off_t back = off_t(max(kk[q] - left + 1, 0)) * (ALONG_K ? off_t(1) : off_t(ld));
			v[q]             = read(p + (off[q] - back * off_t((CPLX ? 2 : 1) * sizeof(double))));
			if (kk[q] >= left)
				v[q] = vd2 { 0.0, 0.0 };
		}
	}
	__device__ inline static vd2 read(vb_gptr p)
	{
		if constexpr (CPLX)
			return *(const __attribute__((address_space(1))) vd2u*)p;
		else
			return vd2 { *(const __attribute__((address_space(1))) double*)p, 0.0 };
	}
	__device__ inline void store(double* lds, const vd2 v[E], int tid) const
	{
#pragma unroll
		for (int q = 0; q < E; ++q) {
			const int e  = tid + kVbThreads * q;
			const int r  = trow(e);
			const int at = ALONG_K ? r * kVbK + 2 * slot(r, kk[q] >> 1) + (kk[q] & 1)
			                       : kk[q] * LDK + r;
			lds[at] = v[q].x;
			if constexpr (CPLX)
				lds[LDS + at] = sign * v[q].y;
		}
	}
	__device__ inline static int slot(int r, int kv) { return kv ^ ((r & 7) ^ ((r >> 3) & 1)); }
	// Element k = 4 g + 2 v + e (e < 2) of row r of a plane.
	__device__ inline static vd2 frag(const double* lds, int r, int g, int v)
	{
		if constexpr (ALONG_K)
			return *reinterpret_cast<const vd2*>(lds + r * kVbK + 2 * slot(r, 2 * g + v));
		const int k = 4 * g + 2 * v;
		return vd2 { lds[k * LDK + r], lds[(k + 1) * LDK + r] };
	}
};

__device__ inline vd4 vb_mma(double a, double b, vd4 c)
{
	return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// AK / BK: op(A)^T's / op(B)^T's rows run along k in memory (A transposed, B not).
template <int T, bool AK, bool BK, bool CPLX, bool WIDE>
__global__ __launch_bounds__(kVbThreads) void vb_gemm_kernel(
    const VbEntry* __restrict__ entries, const VbRun* __restrict__ runs, int nruns, int conja,
    int conjb, int skip, double ar, double ai, double br, double bi, int beta_zero)
{
	using OA          = VbOperand<T, AK, CPLX, WIDE>; // columns of C^T: rows i of C
	using OB          = VbOperand<T, BK, CPLX, WIDE>; // rows of C^T: columns j of C
	constexpr int P   = CPLX ? 2 : 1;
	constexpr int F   = T / 32; // 16 x 16 blocks per wave each way
	__shared__ __attribute__((aligned(16))) double sa[2][P * OA::LDS];
	__shared__ __attribute__((aligned(16))) double sb[2][P * OB::LDS];

	const int     tid = threadIdx.x, lane = tid & 63;
	// Workgroup b is position b / 8 of XCD b % 8's list; its run is the last that starts there or
	// before: 64 candidates at a time, evenly over what is left of the list, so lists of up to 4096
	// runs take two dependent loads.
	const int    pos  = int(blockIdx.x) / kVbXcds;
	const VbRun* list = runs + int64_t(blockIdx.x % kVbXcds) * nruns;
	int          run  = 0;
	for (int end = nruns; end - run > 1;) {
		const int      step  = (end - run + 63) / 64;
		const int      at    = run + lane * step;
		const uint64_t mask  = __ballot(at < end && list[at].first <= pos);
		const int      below = max(__popcll(mask), 1) - 1;
		end                  = min(end, run + (below + 1) * step);
		run += below * step;
	}
	const VbRun rn = list[__builtin_amdgcn_readfirstlane(run)];
	const int   t  = rn.t0 + pos - rn.first;
	if (pos < rn.first || t >= rn.t1)
		return;
	const VbEntry en = entries[rn.entry];
	const int     tm = (en.m + T - 1) / T;
	const int     m0 = (t % tm) * T, n0 = (t / tm) * T;
	const int     wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int     wj = (wave & 1) * (T / 2), wi = (wave >> 1) * (T / 2);
	const int     g = lane >> 4, lr = lane & 15;
	const int     K   = skip ? 0 : en.k; // alpha = 0: A and B are not read

	vd4 re[F][F], im[CPLX ? F : 1][CPLX ? F : 1], rr[CPLX ? F : 1][CPLX ? F : 1];
#pragma unroll
	for (int j = 0; j < F; ++j)
#pragma unroll
		for (int i = 0; i < F; ++i) {
			re[j][i] = vd4 {};
			if constexpr (CPLX) {
				im[j][i] = vd4 {};
				rr[j][i] = vd4 {};
			}
		}
	if (K > 0) {
		OA oa;
		OB ob;
		oa.setup(en.a, en.lda, m0, en.m, conja != 0, tid);
		ob.setup(en.b, en.ldb, n0, en.n, conjb != 0, tid);
		// nf whole chunks go through the registers kVbAhead deep; the last, partial one waits in
		// registers of its own from the start.
		const int nf = K / kVbK, left = K % kVbK;
		vd2       va[kVbAhead][OA::E], vb[kVbAhead][OB::E], ta[OA::E], tb[OB::E];
		// Past the last whole chunk that one is read again (and not used), so that every step has
		// the same loads in flight.
		auto load = [&](int c, vd2* pa, vd2* pb) {
			const int cc = min(c, nf - 1);
			oa.load(cc, pa);
			ob.load(cc, pb);
			// Keeps the groups of loads in order, so that waiting for one leaves the later ones out.
			asm volatile("" ::: "memory");
		};
		auto store = [&](int buf, const vd2* pa, const vd2* pb) {
			oa.store(sa[buf], pa, tid);
			ob.store(sb[buf], pb, tid);
		};
		auto compute = [&](const double* a, const double* b) {
#pragma unroll
			for (int v = 0; v < 2; ++v) {
				vd2 xa[P][F], xb[P][F];
#pragma unroll
				for (int p = 0; p < P; ++p)
#pragma unroll
					for (int f = 0; f < F; ++f) {
						xa[p][f] = OA::frag(a + p * OA::LDS, wi + 16 * f + lr, g, v);
						xb[p][f] = OB::frag(b + p * OB::LDS, wj + 16 * f + lr, g, v);
					}
#pragma unroll
				for (int e = 0; e < 2; ++e)
#pragma unroll
					for (int j = 0; j < F; ++j)
#pragma unroll
						for (int i = 0; i < F; ++i) {
							re[j][i] = vb_mma(xb[0][j][e], xa[0][i][e], re[j][i]);
							if constexpr (CPLX) {
								rr[j][i] = vb_mma(xb[1][j][e], xa[1][i][e], rr[j][i]);
								im[j][i] = vb_mma(xb[1][j][e], xa[0][i][e], im[j][i]);
								im[j][i] = vb_mma(xb[0][j][e], xa[1][i][e], im[j][i]);
							}
						}
			}
		};
		// This wave's LDS accesses are done, then every wave's; loads in flight are not waited for.
		auto barrier = [&]() {
			__builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
			asm volatile("s_barrier" ::: "memory");
		};
		if (left > 0) {
			oa.load_tail(nf, left, ta);
			ob.load_tail(nf, left, tb);
		}
		if (nf > 0) {
#pragma unroll
			for (int u = 0; u < kVbAhead; ++u)
				load(u, va[u], vb[u]);
			store(0, va[0], vb[0]);
			load(kVbAhead, va[0], vb[0]);
			barrier();
			// At the top of a step LDS buffer c % 2 holds chunk c, and chunks c + 1 .. c + kVbAhead
			// are on their way; chunk c + 1 goes to the other buffer, last read before the last
			// barrier.
			int c0 = 0;
			for (; c0 + kVbAhead <= nf; c0 += kVbAhead) {
#pragma unroll
				for (int u = 0; u < kVbAhead; ++u) {
					constexpr int N = kVbAhead;
					compute(sa[u & 1], sb[u & 1]);
					store((u + 1) & 1, va[(u + 1) % N], vb[(u + 1) % N]);
					load(c0 + u + 1 + N, va[(u + 1) % N], vb[(u + 1) % N]);
					barrier();
				}
			}
#pragma unroll
			for (int u = 0; u < kVbAhead - 1; ++u) {
				if (c0 + u < nf) {
					compute(sa[u & 1], sb[u & 1]);
					if (c0 + u + 1 < nf)
						store((u + 1) & 1, va[u + 1], vb[u + 1]);
				}
				barrier();
			}
		}
		if (left > 0) {
			store(0, ta, tb);
			barrier();
			compute(sa[0], sb[0]);
		}
	}
#pragma unroll
	for (int j = 0; j < F; ++j)
#pragma unroll
		for (int r = 0; r < 4; ++r) {
			const int col = n0 + wj + 16 * j + g + 4 * r;
			if (col >= en.n)
				continue;
#pragma unroll
			for (int i = 0; i < F; ++i) {
				const int row = m0 + wi + 16 * i + lr;
				if (row >= en.m)
					continue;
				const int64_t ic = row + int64_t(col) * en.ldc, id = row + int64_t(col) * en.ldd;
				if constexpr (!CPLX) {
					double v = ar * re[j][i][r];
					if (!beta_zero)
						v += br * en.c[ic];
					en.d[id] = v;
				} else {
					const double cr = re[j][i][r] - rr[j][i][r], ci = im[j][i][r];
					double       xr = ar * cr - ai * ci, xi = ar * ci + ai * cr;
					if (!beta_zero) {
						const double p = en.c[2 * ic], q = en.c[2 * ic + 1];
						xr += br * p - bi * q;
						xi += br * q + bi * p;
					}
					en.d[2 * id]     = xr;
					en.d[2 * id + 1] = xi;
				}
			}
		}
}

__global__ __launch_bounds__(kVbThreads) void vb_copy_back_kernel(
    const VbEntry* __restrict__ entries, int nentries, int width)
{
	for (int e = blockIdx.y; e < nentries; e += gridDim.y) {
		const VbEntry en    = entries[e];
		const int64_t total = int64_t(en.m) * en.n * width;
		const int64_t rows  = int64_t(en.m) * width;
		for (int64_t q = int64_t(blockIdx.x) * kVbThreads + threadIdx.x; q < total;
		     q += int64_t(gridDim.x) * kVbThreads)
			const_cast<double*>(en.c)[q % rows + (q / rows) * (int64_t(en.ldc) * width)] =
			    en.d[q % rows + (q / rows) * (int64_t(en.ldd) * width)];
	}
}

template <int T, bool AK, bool BK, bool CPLX>
void go(const VbLaunch& p, const VbEntry* entries, const VbRun* runs, int nruns, int longest,
        hipStream_t s)
{
	auto kern = p.wide ? vb_gemm_kernel<T, AK, BK, CPLX, true> : vb_gemm_kernel<T, AK, BK, CPLX, false>;
	const int skip = p.ar == 0.0 && (!CPLX || p.ai == 0.0);
	hipLaunchKernelGGL(kern, dim3(unsigned(longest) * kVbXcds), dim3(kVbThreads), 0, s, entries,
	                   runs, nruns, int(p.ta == 2), int(p.tb == 2), skip, p.ar, p.ai, p.br, p.bi,
	                   int(p.beta_zero));
}

template <int T, bool CPLX>
void pick(const VbLaunch& p, const VbEntry* entries, const VbRun* runs, int nruns, int longest,
          hipStream_t s)
{
	if (p.ta && p.tb)
		go<T, true, false, CPLX>(p, entries, runs, nruns, longest, s);
	else if (p.ta)
		go<T, true, true, CPLX>(p, entries, runs, nruns, longest, s);
	else if (p.tb)
		go<T, false, false, CPLX>(p, entries, runs, nruns, longest, s);
	else
		go<T, false, true, CPLX>(p, entries, runs, nruns, longest, s);
}

} // namespace

void launch_vb_gemm(const VbLaunch& p, const VbEntry* entries, const VbRun* runs, int nruns,
                    int longest, hipStream_t s)
{
	if (longest <= 0)
		return;
	if (p.cplx) {
		if (p.tile == 32)
			pick<32, true>(p, entries, runs, nruns, longest, s);
		else
			pick<64, true>(p, entries, runs, nruns, longest, s);
	} else {
		if (p.tile == 32)
			pick<32, false>(p, entries, runs, nruns, longest, s);
		else
			pick<64, false>(p, entries, runs, nruns, longest, s);
	}
	DMK_HIP_CHECK(hipGetLastError());
}

void launch_vb_copy_back(const VbEntry* entries, int nentries, bool cplx, hipStream_t s)
{
	if (nentries <= 0)
		return;
	hipLaunchKernelGGL(vb_copy_back_kernel, dim3(64, unsigned(std::min(nentries, 65535))),
	                   dim3(kVbThreads), 0, s, entries, nentries, cplx ? 2 : 1);
	DMK_HIP_CHECK(hipGetLastError());
}

} // namespace dmk
