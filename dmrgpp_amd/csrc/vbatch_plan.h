// Host planning of a variable-size batched GEMM (vbatch.cpp): whether results have to go through a
// workspace, and which tiles each XCD's workgroups take. Linear in the number of entries for the
// batches a program builds (packed operands, sizes in any order); a batch may hold 10^5 of them.
#pragma once

#include "vbatch.h"

#include <algorithm>
#include <cstdint>
#include <numeric>
#include <vector>

namespace dmk {

struct VbRange {
	uintptr_t lo, hi;
	bool      out;
};

// The memory of all outputs and of all inputs (by range: interleaved submatrices count), each
// matrix joined to the one before it where they touch. Packed operands leave two or three ranges,
// which spares sorting 3 x 10^5 of them (14 of 19 ms for a batch of 10^5 8 x 8 products).
inline std::vector<VbRange> vb_ranges(const std::vector<VbEntry>& ents, int ta, int tb, size_t scalar)
{
	std::vector<VbRange> r;
	size_t               last[3] = { SIZE_MAX, SIZE_MAX, SIZE_MAX };
	auto                 add     = [&](int kind, const double* p, int rows, int cols, int ld) {
                const uintptr_t lo = reinterpret_cast<uintptr_t>(p);
                const uintptr_t hi = lo + (size_t(cols - 1) * size_t(ld) + size_t(rows)) * scalar;
                // An input joins the last A or the last B, which often lie in one buffer in turn.
                for (int j : { kind, kind == 0 ? 0 : 3 - kind }) {
                        if (last[j] == SIZE_MAX)
                                continue;
                        VbRange& l = r[last[j]];
                        if (lo <= l.hi && hi >= l.lo) {
                                l.lo       = std::min(l.lo, lo);
                                l.hi       = std::max(l.hi, hi);
                                last[kind] = last[j];
                                return;
                        }
                }
                last[kind] = r.size();
                r.push_back(VbRange { lo, hi, kind == 0 });
	};
	for (const VbEntry& e : ents) {
		add(0, e.c, e.m, e.n, e.ldc);
		if (e.k > 0) {
			add(1, e.a, ta ? e.k : e.m, ta ? e.m : e.k, e.lda);
			add(2, e.b, tb ? e.n : e.k, tb ? e.k : e.n, e.ldb);
		}
	}
	return r;
}

// By lower end. Matrices that were allocated one by one come in any order: large lists by counting, 12
// bits of the address at a time, in half of std::sort's time. A call of 10^5 products of 8 x 8 matrices
// scattered over memory takes 10.2 ms (26.2 sorting every matrix, 14.3 with staged operands), of
// 20000 of 40 x 40 ones 1.5 (3.9, 2.0).
inline void vb_sort_ranges(std::vector<VbRange>& r)
{
	const auto before = [](const VbRange& x, const VbRange& y) { return x.lo < y.lo; };
	if (std::is_sorted(r.begin(), r.end(), before))
		return;
	if (r.size() < 4096) {
		std::sort(r.begin(), r.end(), before);
		return;
	}
	const auto           ends = std::minmax_element(r.begin(), r.end(), before);
	const uintptr_t      base = ends.first->lo, span = ends.second->lo - base;
	std::vector<VbRange> to(r.size());
	std::vector<size_t>  at(4096);
	for (int shift = 0; shift < 64 && (span >> shift) != 0; shift += 12) {
		const auto digit = [&](const VbRange& x) { return ((x.lo - base) >> shift) & 4095; };
		std::fill(at.begin(), at.end(), 0);
		for (const VbRange& x : r)
			++at[digit(x)];
		size_t sum = 0;
		for (size_t& a : at) {
			const size_t n = a;
			a              = sum;
			sum += n;
		}
		for (const VbRange& x : r)
			to[at[digit(x)]++] = x;
		r.swap(to);
	}
}

// Whether any output's memory range meets any input's.
inline bool vb_outputs_meet_inputs(const std::vector<VbEntry>& ents, int ta, int tb, size_t scalar)
{
	std::vector<VbRange> r = vb_ranges(ents, ta, tb, scalar);
	// Outputs and inputs apart as wholes: nothing to sort.
	uintptr_t lo[2] = { UINTPTR_MAX, UINTPTR_MAX }, hi[2] = { 0, 0 };
	for (const VbRange& x : r) {
		lo[x.out] = std::min(lo[x.out], x.lo);
		hi[x.out] = std::max(hi[x.out], x.hi);
	}
	if (hi[0] <= lo[1] || hi[1] <= lo[0])
		return false;
	vb_sort_ranges(r);
	uintptr_t end[2] = { 0, 0 };
	for (const VbRange& x : r) {
		if (x.lo < end[!x.out])
			return true;
		end[x.out] = std::max(end[x.out], x.hi);
	}
	return false;
}

// Which tiles each XCD's workgroups take (workgroup b runs on XCD b % 8): every entry's tiles, the
// longest contractions first, in eight runs, so that neighbouring tiles share an L2; small entries
// go whole to the XCD with the least work. The workgroups find their tiles in these lists, which
// spares the host and the upload the tiles themselves (a few thousand per call).
struct VbRunLists {
	std::vector<VbRun> runs; // kVbXcds lists of nruns
	int                nruns   = 0;
	int64_t            longest = 0;
};

inline VbRunLists vb_list_runs(const std::vector<VbEntry>& ents, int T)
{
	std::vector<int> order(ents.size());
	std::iota(order.begin(), order.end(), 0);
	const auto longer = [&](int x, int y) { return ents[size_t(x)].k > ents[size_t(y)].k; };
	if (!std::is_sorted(order.begin(), order.end(), longer))
		std::stable_sort(order.begin(), order.end(), longer);
	std::vector<VbRun> lists[kVbXcds];
	double             load[kVbXcds]  = {};
	int64_t            count[kVbXcds] = {};
	for (int e : order) {
		const VbEntry& en   = ents[size_t(e)];
		const int64_t  nt   = int64_t((en.m + T - 1) / T) * ((en.n + T - 1) / T);
		const double   cost = double(en.k) + 32.0;
		for (int64_t run = 0, t = 0; t < nt; ++run) {
			const int64_t end = nt < kVbXcds ? nt : nt * (run + 1) / kVbXcds;
			if (end == t)
				continue;
			const int x = int(std::min_element(load, load + kVbXcds) - load);
			lists[x].push_back(VbRun { int32_t(count[x]), e, int32_t(t), int32_t(end) });
			count[x] += end - t;
			load[x] += cost * double(end - t);
			t = end;
		}
	}
	VbRunLists out;
	for (int x = 0; x < kVbXcds; ++x) {
		out.nruns   = std::max(out.nruns, int(lists[x].size()));
		out.longest = std::max(out.longest, count[x]);
	}
	out.runs.assign(size_t(out.nruns) * kVbXcds, VbRun { INT32_MAX, 0, 0, 0 });
	for (int x = 0; x < kVbXcds; ++x)
		std::copy(lists[x].begin(), lists[x].end(), out.runs.begin() + size_t(x) * size_t(out.nruns));
	return out;
}

} // namespace dmk
