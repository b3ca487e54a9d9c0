// CPU test of the batched GEMM's host planning (vbatch_plan.h): the overlap test against every pair
// of matrices, its size for packed operands, and that the XCDs' run lists hold every tile once.
#include "vbatch_plan.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>

namespace {

int g_failed = 0;

void check(bool ok, const char* what)
{
	if (!ok) {
		std::printf("FAILED: %s\n", what);
		++g_failed;
	}
}

double* at(size_t element) { return reinterpret_cast<double*>(0x700000000000 + 8 * element); }

dmk::VbEntry entry(size_t a, size_t b, size_t c, int m, int n, int k, int pad)
{
	dmk::VbEntry e {};
	e.a   = at(a);
	e.b   = at(b);
	e.c   = at(c);
	e.m   = m;
	e.n   = n;
	e.k   = k;
	e.lda = m + pad;
	e.ldb = k + pad;
	e.ldc = m + pad;
	return e;
}

bool meet_by_pairs(const std::vector<dmk::VbEntry>& ents)
{
	auto span = [](const double* p, int rows, int cols, int ld) {
		return std::make_pair(p, p + (size_t(cols) - 1) * size_t(ld) + size_t(rows));
	};
	for (const auto& x : ents)
		for (const auto& y : ents) {
			if (y.k == 0)
				continue;
			const auto c = span(x.c, x.m, x.n, x.ldc);
			for (const auto& in : { span(y.a, y.m, y.k, y.lda), span(y.b, y.k, y.n, y.ldb) })
				if (c.first < in.second && in.first < c.second)
					return true;
		}
	return false;
}

} // namespace

int main()
{
	std::mt19937 rng(1);
	auto         draw = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); };
	int          met  = 0;
	for (int trial = 0; trial < 4000; ++trial) {
		std::vector<dmk::VbEntry> ents;
		const int                 space = 1 << draw(6, 14);
		for (int i = draw(1, 8); i > 0; --i)
			ents.push_back(entry(size_t(draw(0, space)), size_t(draw(0, space)), size_t(draw(0, space)),
			                     draw(1, 5), draw(1, 5), draw(0, 5), draw(0, 2)));
		const bool want = meet_by_pairs(ents);
		met += want;
		check(dmk::vb_outputs_meet_inputs(ents, 0, 0, 8) == want, "overlaps as by pairs");
	}
	check(met > 400 && met < 3600, "both answers occur");

	// 10^5 products of 8 x 8 blocks: A and B in turn in one buffer, C in another, in between.
	std::vector<dmk::VbEntry> many;
	for (size_t i = 0; i < 100000; ++i)
		many.push_back(entry(128 * i, 128 * i + 64, 20000000 + 64 * i, 8, 8, 8, 0));
	check(dmk::vb_ranges(many, 0, 0, 8).size() == 2, "A and B in turn: one range, and C's");
	check(!dmk::vb_outputs_meet_inputs(many, 0, 0, 8), "apart");
	for (size_t i = 0; i < many.size(); ++i) {
		many[i].a = at(64 * i);
		many[i].b = at(8000000 + 64 * i);
	}
	check(dmk::vb_ranges(many, 0, 0, 8).size() == 3, "packed operands: three ranges");
	many[77777].c = many[5].b;
	check(dmk::vb_outputs_meet_inputs(many, 0, 0, 8), "one C in a B among 10^5");

	// 20000 products of matrices allocated one by one, in any order: nothing joins.
	{
		std::vector<size_t> slot(60000);
		for (size_t i = 0; i < slot.size(); ++i)
			slot[i] = i;
		std::shuffle(slot.begin(), slot.end(), rng);
		std::vector<dmk::VbEntry> apart;
		for (size_t i = 0; i < 20000; ++i)
			apart.push_back(entry(4096 * slot[3 * i], 4096 * slot[3 * i + 1], 4096 * slot[3 * i + 2], 40,
			                      40, 40, 0));
		std::vector<dmk::VbRange> r = dmk::vb_ranges(apart, 0, 0, 8);
		check(r.size() == 60000, "matrices with gaps stay apart");
		dmk::vb_sort_ranges(r);
		bool sorted = true;
		for (size_t i = 0; i < r.size(); ++i)
			sorted = sorted && r[i].lo == reinterpret_cast<uintptr_t>(at(4096 * i)) && r[i].hi - r[i].lo == 12800;
		check(sorted, "by lower end, every range once");
		check(!dmk::vb_outputs_meet_inputs(apart, 0, 0, 8), "apart in any order");
		apart[12345].c = apart[54].a + 1599;
		check(dmk::vb_outputs_meet_inputs(apart, 0, 0, 8), "one C at the last element of an A");
	}

	for (int T : { 32, 64 })
		for (int count : { 1, 7, 65, 4097, 40000 }) {
			std::vector<dmk::VbEntry> ents;
			for (int i = 0; i < count; ++i)
				ents.push_back(entry(0, 0, 0, draw(1, 200), draw(1, 200), draw(0, 300), 0));
			const dmk::VbRunLists     l = dmk::vb_list_runs(ents, T);
			std::vector<std::vector<int>> seen(ents.size());
			for (size_t e = 0; e < ents.size(); ++e)
				seen[e].assign(size_t((ents[e].m + T - 1) / T * ((ents[e].n + T - 1) / T)), 0);
			for (int x = 0; x < dmk::kVbXcds; ++x) {
				int32_t pos = 0;
				for (int r = 0; r < l.nruns; ++r) {
					const dmk::VbRun& run = l.runs[size_t(x) * size_t(l.nruns) + size_t(r)];
					if (run.first == INT32_MAX) {
						pos = INT32_MAX;
						continue;
					}
					check(run.first == pos, "a list's runs follow each other");
					pos += run.t1 - run.t0;
					check(pos <= l.longest, "no list is longer than the longest");
					for (int t = run.t0; t < run.t1; ++t)
						++seen[size_t(run.entry)][size_t(t)];
				}
			}
			bool once = true;
			for (const auto& s : seen)
				for (int n : s)
					once = once && n == 1;
			check(once, "every tile once");
		}
	if (g_failed)
		return EXIT_FAILURE;
	std::printf("all checks passed\n");
	return EXIT_SUCCESS;
}
