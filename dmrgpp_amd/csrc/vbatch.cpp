// Variable-size batched GEMM: dmrg_Xgemm_vbatch (GPUPlugin/dmrg_vbatch.cpp:129-652) on FP64
// MFMAs.
//
// The reference expands its groups into per-entry arrays and hands them to MAGMA
// *_vbatched_max_nocheck (or a BLAS loop). Here one launch computes the output tiles of all
// entries straight from the caller's matrices (vbatch_kernels.hip); the host checks the arguments
// and uploads the entries and the XCDs' tile lists (vbatch_plan.h) in one copy. A batch in which some
// C overlaps an operand's memory is computed into a workspace and copied back. The call is
// synchronous, like the reference's.
#include "vbatch.h"

#include "dmk_internal.h"
#include "pool.h"
#include "vbatch_plan.h"

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

namespace dmk {

namespace {

// op code of a BLAS transpose character: 0 = N, 1 = T, 2 = C (conjugate transpose).
int trans_code(char t, const char* which)
{
	switch (t) {
	case 'N':
	case 'n':
		return 0;
	case 'T':
	case 't':
		return 1;
	case 'C':
	case 'c':
		return 2;
	default:
		throw std::invalid_argument(std::string("gemm_vbatch: bad ") + which + " '" + t + "'");
	}
}

} // namespace

void gemm_vbatch(bool cplx, char transa, char transb, const int* m, const int* n, const int* k,
                 const double* alpha, const double* const* a, const int* lda,
                 const double* const* b, const int* ldb, const double* beta, double* const* c,
                 const int* ldc, size_t group_count, const int* group_size)
{
	const int ta = trans_code(transa, "transa");
	const int tb = trans_code(transb, "transb");
	if (group_count == 0)
		return;
	if (!m || !n || !k || !alpha || !a || !lda || !b || !ldb || !beta || !c || !ldc || !group_size)
		throw std::invalid_argument("gemm_vbatch: null argument");
	std::vector<VbEntry> ents;
	size_t             idx = 0;
	for (size_t g = 0; g < group_count; ++g) {
		if (group_size[g] < 0 || m[g] < 0 || n[g] < 0 || k[g] < 0)
			throw std::invalid_argument("gemm_vbatch: negative size in group " + std::to_string(g));
		const int rowsA = ta ? k[g] : m[g];
		const int rowsB = tb ? n[g] : k[g];
		if (lda[g] < std::max(1, rowsA) || ldb[g] < std::max(1, rowsB) || ldc[g] < std::max(1, m[g]))
			throw std::invalid_argument("gemm_vbatch: leading dimension too small in group "
			                            + std::to_string(g));
		for (int i = 0; i < group_size[g]; ++i, ++idx) {
			VbEntry e { a[idx], b[idx], c[idx], c[idx], m[g], n[g], k[g], lda[g], ldb[g], ldc[g],
				    ldc[g], 0 };
			if (e.m == 0 || e.n == 0)
				continue;
			if (!e.c || (e.k > 0 && (!e.a || !e.b)))
				throw std::invalid_argument("gemm_vbatch: null matrix pointer at entry "
				                            + std::to_string(idx));
			ents.push_back(e);
		}
	}
	if (ents.empty())
		return;
	const bool alpha_zero = alpha[0] == 0.0 && (!cplx || alpha[1] == 0.0); // A and B are not read
	for (const VbEntry& e : ents)
		if (!alpha_zero && e.k > kVbMaxK)
			throw std::runtime_error("gemm_vbatch: a contraction is longer than "
			                         + std::to_string(kVbMaxK));
	VbLaunch p {};
	p.cplx      = cplx;
	p.ta        = ta;
	p.tb        = tb;
	p.ar        = alpha[0];
	p.ai        = cplx ? alpha[1] : 0.0;
	p.br        = beta[0];
	p.bi        = cplx ? beta[1] : 0.0;
	p.beta_zero = p.br == 0.0 && p.bi == 0.0;
	// 64 x 64 tiles from four per CU on (half the LDS and operand traffic per product); below, four
	// times as many 32 x 32 ones balance better. Two calls of a transformation step with 32- / 64-wide
	// tiles: m = 2048 (443 and 830 tiles of 64 x 64) 187 / 210 us, m = 4096 (1700 and 3200)
	// 951 / 814 us, m = 6000 2720 / 2177 us.
	double tiles64 = 0;
	for (const VbEntry& e : ents) {
		tiles64 += double((e.m + 63) / 64) * double((e.n + 63) / 64);
		p.wide = p.wide || e.lda > kVbNarrowLd || e.ldb > kVbNarrowLd;
	}
	p.tile = tiles64 < 4 * 256 ? 32 : 64;
	if (tiles64 * double(64 / p.tile) * double(64 / p.tile) > double(0x7fffffff / kVbXcds))
		throw std::runtime_error("gemm_vbatch: batch too large for one launch");
	const VbRunLists lists = vb_list_runs(ents, p.tile);
	const size_t   scalar  = (cplx ? 2 : 1) * sizeof(double);
	const bool     through = !alpha_zero && vb_outputs_meet_inputs(ents, ta, tb, scalar);

	const size_t ebytes = ents.size() * sizeof(VbEntry), rbytes = lists.runs.size() * sizeof(VbRun);
	void*        host = nullptr;
	void*        dev  = nullptr;
	void*        work = nullptr;
	hipStream_t  s    = nullptr;
	auto         give_back = [&] {
                pool_host_free(host);
                pool_device_free(dev);
                pool_device_free(work);
	};
	try {
		if (through) {
			size_t elems = 0;
			for (const VbEntry& e : ents)
				elems += size_t(e.m) * size_t(e.n);
			work = pool_device_alloc(elems * scalar);
			double* at = static_cast<double*>(work);
			for (VbEntry& e : ents) {
				e.d   = at;
				e.ldd = e.m;
				at += size_t(e.m) * size_t(e.n) * (cplx ? 2 : 1);
			}
		}
		host = pool_host_alloc(ebytes + rbytes);
		dev  = pool_device_alloc(ebytes + rbytes);
		std::memcpy(host, ents.data(), ebytes);
		std::memcpy(static_cast<char*>(host) + ebytes, lists.runs.data(), rbytes);
		DMK_HIP_CHECK(hipMemcpyAsync(dev, host, ebytes + rbytes, hipMemcpyHostToDevice, s));
		const VbEntry* d_ents = static_cast<const VbEntry*>(dev);
		const VbRun*   d_runs = reinterpret_cast<const VbRun*>(static_cast<char*>(dev) + ebytes);
		launch_vb_gemm(p, d_ents, d_runs, lists.nruns, int(lists.longest), s);
		if (through)
			launch_vb_copy_back(d_ents, int(ents.size()), cplx, s);
		DMK_HIP_CHECK(hipStreamSynchronize(s));
	} catch (...) {
		(void)hipDeviceSynchronize();
		give_back();
		throw;
	}
	give_back();
}

} // namespace dmk
