// CPU test of the host side of the captured Lanczos steps (lanczos_step.h) on stand-ins for the
// HIP calls it makes: a stream whose last graph launch is still running until somebody waits.
#include "lanczos_step.h"

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
	if (g_failed)
		return EXIT_FAILURE;
	std::printf("all checks passed\n");
	return EXIT_SUCCESS;
}
