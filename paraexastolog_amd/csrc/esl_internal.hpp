// Internal declarations shared by the host API and the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/esl.h"
#include "model.hpp"

#define ESL_HIP(call)                                                                                          \
	do                                                                                                         \
	{                                                                                                          \
		hipError_t e_ = (call);                                                                                \
		if (e_ != hipSuccess)                                                                                  \
		{                                                                                                      \
			(void)hipGetLastError(); /* reported here, and not by the next launch's check too */               \
			throw ::esl::error(e_ == hipErrorOutOfMemory ? ESL_E_OOM : ESL_E_DEVICE,                           \
							   std::string(#call) + ": " + hipGetErrorString(e_) + " (" + __FILE__ + ":" +    \
								   std::to_string(__LINE__) + ")");                                            \
		}                                                                                                      \
	} while (0)

namespace esl {

// Device memory that a context's buffers leave and take again.  hipMalloc and
// hipFree of a few MB map and unmap memory: a model of 20 nodes through the class
// API calls each 85 times, at 35 and 45 us on average 6.8 of its 17.7 ms (10.5 with the
// pool; 15 nodes: 4.3 to 3.8 ms).  A block is reused by work on the same context only: calls on
// one context are serialised on its stream, so what was enqueued on a block comes
// before what its next owner enqueues.  Small blocks cost 1.6 us a pair (115 us
// of the 1.06 ms of a model of 10 nodes).  Blocks above a quarter of the bound
// (of 512 MB) are not kept; the oldest leave when there are more than 512 or the bound is
// exceeded, all when an allocation fails and when the context is destroyed (buffers that
// outlive it are freed directly).
struct buf_pool_t
{
	static constexpr size_t least = 256, most_blocks = 512;
	const size_t bound, largest; // bytes kept, and of one block
	std::weak_ptr<buf_pool_t> other; // the context's other pool
	explicit buf_pool_t(size_t most = (size_t)512 << 20, size_t one = (size_t)128 << 20) : bound(most), largest(one) {}
	struct block_t
	{
		void* p;
		size_t bytes;
	};
	std::mutex m;
	std::vector<block_t> blocks; // oldest first
	size_t held = 0;
	bool closed = false;

	// a kept block of at least `bytes` and at most a quarter more, or {null, 0}
	block_t take(size_t bytes)
	{
		std::lock_guard<std::mutex> g(m);
		size_t best = blocks.size();
		for (size_t i = 0; i < blocks.size(); ++i)
			if (blocks[i].bytes >= bytes && blocks[i].bytes <= bytes + bytes / 4 &&
				(best == blocks.size() || blocks[i].bytes < blocks[best].bytes))
				best = i;
		if (best == blocks.size())
			return { nullptr, 0 };
		const block_t b = blocks[best];
		blocks.erase(blocks.begin() + best);
		held -= b.bytes;
		return b;
	}
	void give(void* p, size_t bytes)
	{
		std::vector<block_t> out;
		{
			std::lock_guard<std::mutex> g(m);
			if (closed || bytes < least || bytes > largest)
				out.push_back({ p, bytes });
			else
			{
				blocks.push_back({ p, bytes });
				held += bytes;
				while (held > bound || blocks.size() > most_blocks)
				{
					out.push_back(blocks.front());
					held -= blocks.front().bytes;
					blocks.erase(blocks.begin());
				}
			}
		}
		for (const block_t& b : out)
			(void)hipFree(b.p);
	}
	// frees what is kept; with `close`, later blocks are freed as they come
	void clear(bool close)
	{
		std::vector<block_t> out;
		{
			std::lock_guard<std::mutex> g(m);
			out.swap(blocks);
			held = 0;
			closed = closed || close;
		}
		for (const block_t& b : out)
			(void)hipFree(b.p);
	}
	// frees what this pool and the other one keep
	void clear_both()
	{
		clear(false);
		if (const auto o = other.lock())
			o->clear(false);
	}
	// hipMalloc, once more without the kept blocks
	hipError_t alloc(void** p, size_t bytes)
	{
		const hipError_t e = hipMalloc(p, bytes);
		if (e != hipErrorOutOfMemory)
			return e;
		(void)hipGetLastError();
		clear_both();
		return hipMalloc(p, bytes);
	}
	~buf_pool_t() { clear(true); }
};

// pool of the context whose call the thread is in (the library's own host threads:
// of their child context); buffers of another context are freed, not given back
inline thread_local std::shared_ptr<buf_pool_t> tl_pool;
// pool that gives its memory back where a call whose buffers do not come from it runs out
inline thread_local std::shared_ptr<buf_pool_t> tl_spare;
struct pool_scope_t
{
	std::shared_ptr<buf_pool_t>& at;
	std::shared_ptr<buf_pool_t> before;
	explicit pool_scope_t(std::shared_ptr<buf_pool_t> p, std::shared_ptr<buf_pool_t>& where = tl_pool)
		: at(where), before(std::move(where))
	{
		at = std::move(p);
	}
	~pool_scope_t() { at = std::move(before); }
};

// Owning device buffer.
template <typename T>
struct dbuf
{
	T* p = nullptr;
	size_t n = 0;
	size_t bytes = 0; // of the allocation
	std::shared_ptr<buf_pool_t> pool;
	dbuf() = default;
	dbuf(const dbuf&) = delete;
	dbuf& operator=(const dbuf&) = delete;
	dbuf(dbuf&& o) noexcept : p(o.p), n(o.n), bytes(o.bytes), pool(std::move(o.pool)) { o.p = nullptr, o.n = o.bytes = 0; }
	dbuf& operator=(dbuf&& o) noexcept
	{
		reset();
		p = o.p, n = o.n, bytes = o.bytes, pool = std::move(o.pool);
		o.p = nullptr, o.n = o.bytes = 0;
		return *this;
	}
	~dbuf() { reset(); }
	void reset()
	{
		if (p && pool && (!tl_pool || tl_pool == pool))
			pool->give(p, bytes);
		else if (p)
			(void)hipFree(p);
		p = nullptr, n = bytes = 0;
		pool.reset();
	}
	// grows only; contents are not preserved
	void ensure(size_t count)
	{
		if (count <= n && p)
			return;
		reset();
		if (count == 0)
			count = 1;
		bytes = count * sizeof(T);
		pool = tl_pool;
		if (pool)
		{
			const auto b = pool->take(bytes);
			if (b.p)
			{
				p = static_cast<T*>(b.p);
				n = count;
				bytes = b.bytes;
				return;
			}
		}
		void* q = nullptr;
		const hipError_t e = pool		? pool->alloc(&q, bytes)
							 : tl_spare ? tl_spare->alloc(&q, bytes)
										: hipMalloc(&q, bytes);
		p = static_cast<T*>(q);
		if (e != hipSuccess)
		{
			p = nullptr;
			pool.reset();
		}
		ESL_HIP(e);
		n = count;
	}
	T* get() const { return p; }
};

// Device form of the rules: per node {k, input offset, table bit offset}.
struct rule_dev_t
{
	int32_t k;
	int32_t in_off;
	int32_t tab_off; // in bits
	int32_t pad;
};

struct graph_t;

// Per-kernel timing with HIP events on the context stream (off by default).
struct kstat_t
{
	int64_t launches = 0;
	double ms = 0.0;
	double bytes = 0.0; // algorithmic bytes summed over the launches
};

struct prof_t
{
	bool on = false;
	struct pending_t
	{
		const char* name;
		hipEvent_t a, b;
		double bytes;
	};
	std::vector<pending_t> pending;
	std::vector<hipEvent_t> pool;
	size_t used = 0;
	std::vector<std::pair<std::string, kstat_t>> stats;
	// while a HIP graph is being captured: its event pairs go to the graph's owner
	std::vector<hipEvent_t>* capture_events = nullptr;
	std::vector<pending_t>* capture_pending = nullptr;

	hipEvent_t next_event()
	{
		if (capture_events)
		{
			hipEvent_t e;
			if (hipEventCreate(&e) != hipSuccess)
				throw error(ESL_E_DEVICE, "hipEventCreate failed");
			capture_events->push_back(e);
			return e;
		}
		if (used == pool.size())
		{
			hipEvent_t e;
			if (hipEventCreate(&e) != hipSuccess)
				throw error(ESL_E_DEVICE, "hipEventCreate failed");
			pool.push_back(e);
		}
		return pool[used++];
	}
	kstat_t& stat(const std::string& name)
	{
		for (auto& p : stats)
			if (p.first == name)
				return p.second;
		stats.emplace_back(name, kstat_t{});
		return stats.back().second;
	}
	// books the event pairs of one completed launch sequence (the stream must be idle)
	void book(const std::vector<pending_t>& list)
	{
		for (auto& p : list)
		{
			float ms = 0;
			if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess)
			{
				kstat_t& k = stat(p.name);
				k.launches++;
				k.ms += ms;
				k.bytes += p.bytes;
			}
			else
				(void)hipGetLastError(); // an untimed pair is skipped, not left as the next call's error
		}
	}
	void flush()
	{
		book(pending);
		pending.clear();
		used = 0;
	}
	~prof_t()
	{
		for (auto e : pool)
			(void)hipEventDestroy(e);
	}
};

constexpr int flag_words = 64, live_words = 2 * 1024;

struct ctx_t
{
	int device = 0;
	int lds_per_block = 65536; // dynamic + static LDS a workgroup may use on this device
	hipStream_t stream = nullptr;
	std::string last_error;
	hipEvent_t ev[16] = {};
	// reusable scratch
	dbuf<uint8_t> scratch_a, scratch_b;
	dbuf<int32_t> flags;	// small device counters / flags
	dbuf<int32_t> scan_sums; // block sums of exclusive_scan_i32
	int32_t* h_flags = nullptr; // pinned mirror
	int32_t* h_live = nullptr;	// pinned, after the mirror: the device-wide solver's sets, twice
	// pinned staging of the per-set outputs of a launch, read back in one copy
	// (allocated with the context: calls that may not allocate use it too)
	unsigned char* h_stage = nullptr;
	size_t h_stage_bytes = 0;
	prof_t prof;
	std::shared_ptr<buf_pool_t> pool = std::make_shared<buf_pool_t>();
	// Pool of device-wide solves' workspaces, with a bound of its own, as they are large: 0.6 GB
	// for 16 sets of 524,288 unknowns, 2.5 GB for the two device-wide plans of a batch of eight
	// networks.  Allocated and freed by each call they took 0.6 of 25 and 4 of 65 ms.  A host
	// thread's context shares the pool of the context that it works for.
	std::shared_ptr<buf_pool_t> wide = std::make_shared<buf_pool_t>((size_t)2 << 30, (size_t)512 << 20);
	bool wide_shared = false; // with another context
	ctx_t()
	{
		pool->other = wide;
		wide->other = pool;
	}
	// forked streams (default priority) and fork/join events for plans solved concurrently
	std::vector<hipStream_t> aux;
	std::vector<hipEvent_t> aux_ev;
	// stream (default priority) and fork/join events of a plan's final-vector fill
	hipStream_t fill_s = nullptr;
	hipEvent_t fill_ev[2] = {};
	// captured sequence of the last concurrent multi-plan solve (owned by solve.hip)
	void* multi = nullptr;
	void (*multi_free)(void*) = nullptr;
	// device address of the library's static scratch array on this device (noalloc_init)
	void* noalloc_scratch = nullptr;
	double wall_khz = 100000.0; // rate of the device wall clock (wall_clock64) in kHz
};

// size of the static device scratch behind esl_plan_solve_noalloc, and the
// device indices it keeps an address for
constexpr size_t noalloc_scratch_bytes = (size_t)64 << 20;
constexpr int max_devices = 64;

// Appends an event-record node to the graph being captured on `s`, after the
// nodes captured so far, and makes it the dependency of what follows.
inline void record_event_node(hipStream_t s, hipEvent_t e)
{
	hipStreamCaptureStatus st;
	unsigned long long id = 0;
	hipGraph_t g = nullptr;
	const hipGraphNode_t* deps = nullptr;
	size_t nd = 0;
	ESL_HIP(hipStreamGetCaptureInfo_v2(s, &st, &id, &g, &deps, &nd));
	if (st != hipStreamCaptureStatusActive)
		throw error(ESL_E_STATE, "stream is not capturing");
	hipGraphNode_t node;
	ESL_HIP(hipGraphAddEventRecordNode(&node, g, deps, nd, e));
	ESL_HIP(hipStreamUpdateCaptureDependencies(s, &node, 1, hipStreamSetCaptureDependencies));
}

// Launch `launch` (a lambda issuing one kernel on c.stream); with profiling on,
// bracket it with events and book `bytes` algorithmic bytes under `name`.
template <typename F>
inline void timed_launch(ctx_t& c, const char* name, double bytes, F&& launch)
{
	if (!c.prof.on)
	{
		launch();
		return;
	}
	hipEvent_t a = c.prof.next_event(), b = c.prof.next_event();
	if (c.prof.capture_pending)
	{
		// an hipEventRecord captured from the stream cannot be timed on replay;
		// explicit event-record nodes can
		record_event_node(c.stream, a);
		launch();
		record_event_node(c.stream, b);
		c.prof.capture_pending->push_back({ name, a, b, bytes });
		return;
	}
	ESL_HIP(hipEventRecord(a, c.stream));
	launch();
	ESL_HIP(hipEventRecord(b, c.stream));
	c.prof.pending.push_back({ name, a, b, bytes });
	if (c.prof.pending.size() > 4096)
	{
		ESL_HIP(hipStreamSynchronize(c.stream));
		c.prof.flush();
	}
}

struct solution_t
{
	bool valid = false;
	std::vector<int32_t> term_indptr, term_indices;
	std::vector<double> term_data;
	std::vector<int32_t> nonterm_indptr, nonterm_indices;
	std::vector<double> nonterm_data;
};

struct graph_t
{
	int N = 0;
	int64_t n = 0, nnz = 0;
	std::vector<double> rates; // rates given to esl_table_build (zero pattern)
	uint32_t up_ok = 0, down_ok = 0;

	// table
	dbuf<rule_dev_t> rules;
	dbuf<int32_t> rule_inputs;
	dbuf<uint32_t> rule_tables;
	dbuf<uint32_t> mask;   // n: bit i set iff s -> s ^ (1 << i)
	dbuf<int32_t> indptr;  // n + 1
	dbuf<int32_t> rows;	   // nnz (targets)
	dbuf<int32_t> cols;	   // nnz (sources)

	// graph
	bool reorganized = false;
	int64_t S = 0, T = 0, n_t = 0;
	int32_t H = 0;
	dbuf<int32_t> scc;		 // n: canonical SCC id (minimum vertex)
	dbuf<int32_t> height;	 // n: height of the vertex's SCC
	dbuf<int32_t> reordered; // n
	dbuf<int32_t> offsets;	 // S + 1
	dbuf<int32_t> rank;		 // n: position of the vertex's SCC in the canonical SCC order
	std::vector<int32_t> h_offsets; // host copy of offsets (S + 1)

	double stage_ms[2] = { 0, 0 };
	// graph stage counters: passes over the flip masks, SCC rounds, host round trips
	int64_t mask_passes = 0, scc_rounds = 0, host_syncs = 0;
	solution_t sol;
};

// ---- kernel launchers (defined in the .hip files) ----
void table_build(ctx_t& c, graph_t& g, const model_t& m);
void device_copy(ctx_t& c, void* dst, const void* src, size_t bytes);
void graph_reorganize(ctx_t& c, graph_t& g);
void graph_import(ctx_t& c, graph_t& g, const int32_t* h_reordered, const int32_t* h_offsets, int64_t S, int64_t T);

struct solve_args_t
{
	const double* d_rates; // [n_sets][2N]
	const double* d_x0;	   // [n] shared
	double* d_final;	   // [n_sets][n]
	int n_sets;
	esl_solve_opts opts;
};
void solve_run(ctx_t& c, graph_t& g, const solve_args_t& a, esl_solve_report& rep);
// rate-independent solve plans (solve.hip)
void* plan_create(ctx_t& c, graph_t& g, const double* d_x0);
void plan_destroy(void* p);
void plan_solve(ctx_t& c, void* p, int B, const double* d_rates, double* d_final, const esl_solve_opts& o,
				esl_solve_report& rep);
void plan_info(const void* p, int64_t info[8]);
void plan_solve_many(ctx_t& c, int np, void* const* plans, const int* B, const double* const* d_rates,
					 double* const* d_final, const esl_solve_opts& o, esl_solve_report* reps);
void plan_autotune(ctx_t& c, void* p, int B, const double* d_rates, double* d_final, const esl_solve_opts& o,
				   int32_t choice[2], double* best_ms);
void plan_gather_terminal(ctx_t& c, const void* p, int B, const double* d_final, double* d_out);
void plan_set_schedule(void* p, int path, int restart);
void plan_set_results(const void* p, int B, double* res, int32_t* its, int32_t* method);
void plan_set_times(const void* p, int B, double wall_khz, double* start_ms, double* end_ms);
// pinned staging buffer of a context for per-set outputs (32 B per set with the
// clocks: batches of up to 8192 sets in one copy)
constexpr size_t stage_bytes = 256 * 1024;
// the plan solve whose buffers are slices of the static scratch (no allocation)
void noalloc_init(ctx_t& c); // once per device, with that device current
void plan_solve_noalloc(ctx_t& c, void* p, int B, const double* d_rates, double* d_final, const esl_solve_opts& o,
						esl_solve_report& rep);
// the implementation object behind an esl_ctx handle (defined in esl_api.cpp)
ctx_t& ctx_impl(esl_ctx* ctx);
// solution_term / solution_nonterm of one rate set into g.sol (reference layout)
void solution_full(ctx_t& c, graph_t& g, const double* d_rates, const esl_solve_opts& opts);

// device scan helper: out[i] = sum_{j<i} in[j] (exclusive), out[n] = total; in/out int32
void exclusive_scan_i32(ctx_t& c, const int32_t* in, int32_t* out, int64_t n);

} // namespace esl
