// CPU test of the host side of the captured Lanczos steps (lanczos_step.h) on stand-ins for the
// HIP calls it makes: a stream whose last graph launch is still running until somebody waits.
#include "lanczos_step.h"

#include <cstdint>
#include <cstdio>
#include <cstdlib>

namespace {

bool g_running   = false; // the stream has unfinished work
int  g_destroyed = 0;
int  g_failed    = 0;

void check(bool ok, const char* what)
{
	if (!ok) {
		std::printf("FAILED: %s\n", what);
		++g_failed;
	}
}

} // namespace

extern "C" {
hipError_t hipStreamSynchronize(hipStream_t)
{
	g_running = false;
	return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t)
{
	check(!g_running, "an executable graph was destroyed while its launch was running");
	++g_destroyed;
	return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t)
{
	check(!g_running, "a graph was destroyed while its launch was running");
	++g_destroyed;
	return hipSuccess;
}
}

int main()
{
	// The solve's end, an exception between two steps, and a capture that failed half way while the
	// first step runs: none of the graphs goes before the stream's work is done.
	for (int captured = 0; captured <= 3; ++captured) {
		g_running   = true;
		g_destroyed = 0;
		try {
			dmk::StepGraphs sg(nullptr);
			for (int i = 0; i < captured; ++i) {
				sg.g[i] = reinterpret_cast<hipGraph_t>(0x100 + i);
				sg.e[i] = reinterpret_cast<hipGraphExec_t>(0x200 + i);
			}
			if (captured < 3)
				throw 1;
		} catch (int) {
		}
		check(g_destroyed == 2 * captured, "every graph is destroyed once");
		check(!g_running, "the stream's work is done when the owner is gone");
	}
	// Every value is a report, whatever its bits, and comes back: numbers as they were, any NaN as
	// a NaN.
	const uint64_t words[] = { 0, 1, 0x3ff0000000000000, 0xbff8000000000001, 0x7fefffffffffffff,
		                   0x7ff0000000000000, 0xfff0000000000000, 0x7ff8000000000000,
		                   0xfff8000000000000, 0x7fffffffffffffff, 0xfffffffffffffffe, ~uint64_t(0) };
	for (const uint64_t w : words) {
		const double v = dmk::report_value(w);
		uint64_t     r[2];
		for (int first = 0; first < 2; ++first) {
			dmk::clear_report(r);
			check(!dmk::report_there(r), "a cleared report is not there");
			r[first] = dmk::report_word(v);
			check(!dmk::report_there(r), "half a report is not there");
			r[1 - first] = dmk::report_word(1.5);
			check(dmk::report_there(r), "a report of any two values is there");
			const double back = dmk::report_value(r[first]);
			check(v != v ? back != back : dmk::report_word(back) == w, "a value comes back");
		}
	}
	if (g_failed)
		return EXIT_FAILURE;
	std::printf("all checks passed\n");
	return EXIT_SUCCESS;
}
