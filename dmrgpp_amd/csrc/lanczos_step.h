// Host side of the captured Lanczos steps (lanczos.cpp): the step report and the owner of the graphs.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

namespace dmk {

// The step report in pinned memory: alpha_j and beta_{j+1}, each one word that the last kernel of a
// step stores whole and the host polls for, instead of waiting for the stream: a stream wait and
// the next launch after it left the chip idle for 35 to 50 us per step.
//
// A word that is not there yet is all ones. That is a NaN, and arithmetic hands a NaN's payload on
// (memory filled with 0xff as the start vector), so NaNs are reported as the one quiet NaN below.
constexpr uint64_t kNoReport = ~uint64_t(0);

__host__ __device__ inline uint64_t report_word(double v)
{
	if (v != v)
		return 0x7ff8000000000000u;
	uint64_t w = 0;
	memcpy(&w, &v, sizeof(w));
	return w;
}

inline void clear_report(uint64_t* report)
{
	for (int i = 0; i < 2; ++i)
		__atomic_store_n(report + i, kNoReport, __ATOMIC_RELEASE);
}

inline bool report_there(const uint64_t* report)
{
	return __atomic_load_n(report, __ATOMIC_ACQUIRE) != kNoReport
	       && __atomic_load_n(report + 1, __ATOMIC_ACQUIRE) != kNoReport;
}

inline double report_value(uint64_t word)
{
	double v = 0;
	memcpy(&v, &word, sizeof(v));
	return v;
}

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
