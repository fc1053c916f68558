// Fixpoints over the N-cube of states, shared by the graph stage and the plan builder:
// passes enqueued in groups, and the unrolled loops over a state's neighbours.
#pragma once

#include <algorithm>

#include "common.hip.hpp"
#include "esl_internal.hpp"

namespace esl {

// Moves along the high bits 6 .. N-1 read the neighbouring sub-cubes.  The
// kernels below take them in a fully unrolled loop of HMAX steps, step j on
// bit min(6 + j, N - 1) and counted only while 6 + j < N, so all of a lane's
// neighbour loads are in flight before the first is used (a loop bounded by
// the run-time N waits for each load in turn: one memory latency per bit).
// HMAX is the smallest of 8, 16, 26 that covers N - 6 (0 below N = 7).
__device__ __forceinline__ int high_bit(int j, int N) { return 6 + j < N ? 6 + j : N - 1; }

// Fixpoint passes are enqueued in groups without waiting for the host; a
// pass whose predecessor changed nothing (prev[0] == 0) returns at once.
__device__ __forceinline__ bool converged(const int32_t* prev) { return prev && prev[0] == 0; }

// Runs a fixpoint pass in groups of launches with one host round trip per
// group: pass p of a group reports a change in its own flag slot; the first pass
// that changed nothing ends the loop (the passes after it in its group return
// at once, seeing their predecessor's flag clear).  pass(flag, prev) launches
// one pass (prev: the previous pass's flag, null for a group's first).  The
// first group has `hint` passes (what the same fixpoint needed last time, plus
// one), later groups `group`; hint is updated to the passes used plus one.
struct fixpoint_t
{
	int passes, syncs;
};
template <typename F>
fixpoint_t fixpoint(ctx_t& c, int& hint, int group, int max_passes, const char* what, F&& pass)
{
	constexpr int base = 8, slots = 16; // flag slots base .. base + slots - 1
	int32_t* d = c.flags.get() + base;
	int syncs = 0;
	for (int done = 0;;)
	{
		++syncs;
		const int gsz = std::min(slots, std::max(2, done ? group : hint));
		ESL_HIP(hipMemsetAsync(d, 0, gsz * sizeof(int32_t), c.stream));
		for (int p = 0; p < gsz; ++p)
			pass(d + p, p ? d + p - 1 : nullptr);
		ESL_HIP(hipMemcpyAsync(c.h_flags + base, d, gsz * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
		ESL_HIP(hipStreamSynchronize(c.stream));
		for (int p = 0; p < gsz; ++p)
			if (!c.h_flags[base + p])
			{
				hint = done + p + 2;
				return { done + p + 1, syncs };
			}
		done += gsz;
		if (done > max_passes)
			throw error(ESL_E_DEVICE, std::string(what) + " did not converge");
	}
}

// the unrolled width of the high-bit loops for N state bits
inline int hmax_for(int N) { return N <= 6 ? 0 : N <= 14 ? 8 : N <= 22 ? 16 : 26; }

#define ESL_HMAX_DISPATCH(N, KERNEL, ...)                                                                              \
	switch (hmax_for(N))                                                                                               \
	{                                                                                                                  \
	case 0:                                                                                                            \
		KERNEL<0>__VA_ARGS__;                                                                                          \
		break;                                                                                                         \
	case 8:                                                                                                            \
		KERNEL<8>__VA_ARGS__;                                                                                          \
		break;                                                                                                         \
	case 16:                                                                                                           \
		KERNEL<16>__VA_ARGS__;                                                                                         \
		break;                                                                                                         \
	default:                                                                                                           \
		KERNEL<26>__VA_ARGS__;                                                                                         \
		break;                                                                                                         \
	}

} // namespace esl
