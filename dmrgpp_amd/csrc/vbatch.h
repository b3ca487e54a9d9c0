// Variable-size batched GEMM over caller pointers (the dmrg_Xgemm_vbatch boundary of the
// reference plugin, GPUPlugin/dmrg_vbatch.cpp:129-652).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace dmk {

// One product D = alpha op(A) op(B) + beta C (column major; complex scalars interleaved, leading
// dimensions in scalars). D is C, or a workspace where C overlaps an operand.
struct VbEntry {
	const double* a;
	const double* b;
	const double* c;
	double*       d;
	int32_t       m, n, k;
	int32_t       lda, ldb, ldc, ldd;
	int32_t       pad;
};

// Output tiles [t0, t1) of an entry (column major over its tile grid), which sit at positions
// first, first + 1, ... of one XCD's list.
struct VbRun {
	int32_t first;
	int32_t entry;
	int32_t t0;
	int32_t t1;
};

struct VbLaunch {
	bool   cplx;
	int    ta, tb;   // 0 N, 1 T, 2 C
	int    tile;     // 32 or 64
	bool   wide;     // 64-bit operand offsets (leading dimensions past kVbNarrowLd)
	double ar, ai, br, bi;
	bool   beta_zero;
};

// Largest leading dimension whose byte offsets within a tile fit 32 bits (64 rows, 16 bytes).
constexpr int kVbNarrowLd = 1 << 21;

constexpr int kVbXcds = 8;

// Longest contraction that the entry points take.
constexpr int kVbMaxK = 1 << 21;

// runs: eight lists of nruns each, by position (filled up with first = INT32_MAX); `longest`
// positions in the longest list.
void launch_vb_gemm(const VbLaunch& p, const VbEntry* entries, const VbRun* runs, int nruns,
                    int longest, hipStream_t s);
// C = D for every entry (the workspace results of overlapping batches).
void launch_vb_copy_back(const VbEntry* entries, int nentries, bool cplx, hipStream_t s);

// C_e = alpha op(A_e) op(B_e) + beta C_e for every entry e of every group (m, n, k, lda, ldb,
// ldc per group; pointers per entry, device memory, expanded in group order). cplx selects
// interleaved complex scalars (alpha, beta then point to (re, im) pairs). Synchronous. k is at most
// kVbMaxK unless alpha is 0.
void gemm_vbatch(bool cplx, char transa, char transb, const int* m, const int* n, const int* k,
                 const double* alpha, const double* const* a, const int* lda,
                 const double* const* b, const int* ldb, const double* beta, double* const* c,
                 const int* ldc, size_t group_count, const int* group_size);

} // namespace dmk
