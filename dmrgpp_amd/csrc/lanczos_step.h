// Host side of the captured Lanczos steps (lanczos.cpp): the owner of their graphs.
#pragma once

#include <hip/hip_runtime.h>

namespace dmk {

// The three captured phase graphs of one decomposition (ring roles rotate with period 3). They go
// only after the stream's work is done: the solve stops waiting when a step's two scalars have
// arrived, while that step's last kernel may still be writing vectors, and an exception can leave
// with the first step or a captured one still running. One wait per solve, on every way out.
struct StepGraphs {
	hipStream_t    stream;
	hipGraph_t     g[3] = { nullptr, nullptr, nullptr };
	hipGraphExec_t e[3] = { nullptr, nullptr, nullptr };

	explicit StepGraphs(hipStream_t s) : stream(s) { }
	StepGraphs(const StepGraphs&)            = delete;
	StepGraphs& operator=(const StepGraphs&) = delete;
	~StepGraphs()
	{
		(void)hipStreamSynchronize(stream);
		for (int i = 0; i < 3; ++i) {
			if (e[i])
				(void)hipGraphExecDestroy(e[i]);
			if (g[i])
				(void)hipGraphDestroy(g[i]);
		}
	}
};

} // namespace dmk
