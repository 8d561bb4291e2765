// Host side of the register-resident PCG (resident.h): which systems it takes,
// its launches for one system, and the fall-back to the streaming kernels.

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <optional>

#include "resident.h"

namespace bfmx {

using namespace resident;

namespace {

constexpr int64_t kPerLaunch = 8192;    // iterations of one launch at most (some 0.1 s)

// The exchange words of a launch start at number 0 (the vector words' four
// buffers, nw words each, and the all-gather slots).
__global__ __launch_bounds__(kBlock) void k_clear(View V, int64_t nw, int64_t nslots) {
	int64_t const i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
	if (i < nw) {
		V.w[0][i] = V.w[1][i] = V.w[2][i] = V.w[3][i] = 0;
	}
	if (i < nslots) {
		V.slots[i] = 0;
	}
	if (i == 0) {
		*V.gave_up = 0;
	}
}

// Polls of one wait (tests let waits run out early).
uint32_t poll_limit() {
	const char* e = std::getenv("BFMX_RESIDENT_POLLS");
	return e && std::atoi(e) > 0 ? static_cast<uint32_t>(std::atoi(e)) : kSpinLimit;
}

template <typename MT, int W, int PRE, int NT, bool LEAN>
__global__ __launch_bounds__(NT) void k_resident_pcg(View V, uint32_t polls, int mode, double rtol2,
                                                     double delta2, int64_t stop, Scalars* __restrict__ S) {
	extern __shared__ __align__(16) double dyn[];
	__shared__ Shared sh;
	if (threadIdx.x == 0) {
		sh.polls = polls;
	}
	Run R;
	if (mode == 2) {
		R.rz = S->rz;
		R.rr = S->rr;
		R.bb = S->bb;
		R.tol2 = S->tol2;
		R.beta = S->beta;
		R.rr_true = S->rr_true;
		R.rr_ref = S->rr_ref;
		R.rr_best = S->rr_best;
		R.pq = S->pq;
		R.iter = S->iter;
		R.stall = S->stall;
		R.checking = S->checking;
		R.updates = S->updates;
		R.checks = S->updates - 1;
	}
	run_pcg<MT, W, PRE, NT, LEAN>(V, blockIdx.x, gridDim.x, mode, rtol2, delta2, stop, false, sh,
	                        reinterpret_cast<resident::dbl2*>(dyn), R);
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		S->rz = R.rz;
		S->rr = R.rr;
		S->bb = R.bb;
		S->tol2 = R.tol2;
		S->beta = R.beta;
		S->rr_true = R.rr_true;
		S->rr_ref = R.rr_ref;
		S->rr_best = R.rr_best;
		S->pq = R.pq;
		S->iter = R.iter;
		S->done = R.status;
		S->stall = R.stall;
		S->checking = R.checking;
		S->updates = R.updates;
	}
}

typedef void (*PcgKernel)(View, uint32_t, int, double, double, int64_t, Scalars*);

template <typename MT, int W, int PRE>
PcgKernel pick_threads(int nt) {
	return nt == 512 ? k_resident_pcg<MT, W, PRE, 512, false> : k_resident_pcg<MT, W, PRE, 1024, false>;
}

template <typename MT, int W>
PcgKernel pick_precond(int pre, int nt) {
	return pre == BFMX_PRECOND_JACOBI ? pick_threads<MT, W, BFMX_PRECOND_JACOBI>(nt)
	                                  : pick_threads<MT, W, BFMX_PRECOND_BLOCK_JACOBI>(nt);
}

// no_scratch: a kernel that spills no register.
PcgKernel pick(bool mixed, int width, int pre, int nt, bool no_scratch) {
	if (no_scratch && !mixed && pre == BFMX_PRECOND_BLOCK_JACOBI && nt == 1024) {
		return width <= 7 ? k_resident_pcg<double, 7, BFMX_PRECOND_BLOCK_JACOBI, 1024, true>
		                  : k_resident_pcg<double, 9, BFMX_PRECOND_BLOCK_JACOBI, 1024, true>;
	}
	if (mixed) {
		return width <= 7 ? pick_precond<float, 7>(pre, nt) : pick_precond<float, 9>(pre, nt);
	}
	return width <= 7 ? pick_precond<double, 7>(pre, nt) : pick_precond<double, 9>(pre, nt);
}

// The kernel may be launched with lds bytes of dynamic LDS. The limit belongs to
// the kernel, not to the launch: always the same one, the CU's 160 KB without
// Shared and the batch kernel's word, so that threads do not lower it for each
// other.
int allow_lds(const void* kernel, size_t lds) {
	constexpr int kMost = 160 * 1024 - 2048;
	static_assert(sizeof(Shared) + 64 <= 2048 &&
	              kMaxWindow * sizeof(resident::dbl2) + fixed_bytes<double, kMaxWidth, kRows>() <= kMost);
	if (lds > 48 * 1024) {
		BFMX_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kMost));
	}
	return BFMX_OK;
}

// LDS bytes beside the window.
int fixed(bool mixed, int width, int nt) {
	return mixed || nt <= 512 ? 0 : width <= 7 ? fixed_bytes<double, 7, 1024>() : fixed_bytes<double, 9, 1024>();
}

}  // namespace

namespace resident {

int compute_units(int device) {
	int cus = 0;
	return hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess ? cus : 0;
}

namespace {

CuBudget& budget_of(int device) {
	static std::mutex m;
	// never destroyed: threads may still hold shares while the process exits
	static auto* budgets = new std::map<int, CuBudget>;
	std::lock_guard<std::mutex> const lock(m);
	return budgets->try_emplace(device, compute_units(device)).first->second;
}

}  // namespace

ClusterLock::ClusterLock(int device, int64_t workgroups)
    : m_budget(budget_of(device)), m_share(CuBudget::share(workgroups)) {
	m_budget.take(m_share);
}

ClusterLock::~ClusterLock() {
	m_budget.give(m_share);
}

int window_of(const bfmx_system* s, int64_t G, int threads) {
	int64_t const n = s->n_nodes;
	if (n == 0 || G > kMaxGroup || (n + G - 1) / G > threads) {
		return 0;
	}
	if (*std::max_element(s->row_len.begin(), s->row_len.end()) > kMaxWidth) {
		return 0;
	}
	int64_t const rows = ((n + G - 1) / G + 63) / 64 * 64;
	int32_t widest = 0;
	for (int64_t r0 = 0; r0 < n; r0 += rows) {
		int64_t const r1 = std::min(n, r0 + rows);
		int32_t lo = static_cast<int32_t>(r0), hi = static_cast<int32_t>(r1 - 1);
		for (int64_t i = r0; i < r1; i++) {   // sorted rows
			lo = std::min(lo, s->adj[s->adj_ptr[i]]);
			hi = std::max(hi, s->adj[s->adj_ptr[i + 1] - 1]);
		}
		widest = std::max(widest, hi - lo + 1);
	}
	return widest <= kMaxWindow ? widest : 0;
}

}  // namespace resident

int resident_pcg(bfmx_system* s, int precond, bool mixed, double rtol2, double delta2, int64_t cap, bool warm,
                 bool no_scratch, Scalars* out, bool* ran) {
	*ran = false;
	const char* e = std::getenv("BFMX_RESIDENT");
	if ((e && e[0] == '0') || s->n_conv_seg > 0 || (precond != BFMX_PRECOND_JACOBI && precond != BFMX_PRECOND_BLOCK_JACOBI)) {
		return BFMX_OK;
	}
	if (std::chrono::steady_clock::now() < s->res_retry) {
		return BFMX_OK;
	}
	if (s->res_groups < 0) {
		int64_t const groups = (s->n_nodes + kRows - 1) / kRows;
		s->res_window = groups <= compute_units(s->device) ? window_of(s, groups) : 0;
		s->res_groups = 0;
		if (s->res_window > 0) {
			s->res_groups = static_cast<int>(groups);
			s->res_width = *std::max_element(s->row_len.begin(), s->row_len.end());
		}
	}
	int const G = s->res_groups;
	if (G == 0) {
		return BFMX_OK;
	}
	hipStream_t const st = s->stream;
	int64_t const n = s->n_nodes;
	auto words = [](double* p) { return reinterpret_cast<u64*>(p); };
	View V{s->d_slice_ptr, s->d_col, s->d_diag_blk, s->d_val, s->d_val32, s->d_bsolve, s->d_x,
	       {words(s->d_r), words(s->d_z), words(s->d_q), words(s->d_p[0])}, words(s->d_p[1]), s->d_dinv,
	       &s->d_scal->gave_up, n};
	int const nt = n <= 512 ? 512 : 1024;
	PcgKernel const kernel = pick(mixed, s->res_width, precond, nt, no_scratch);
	size_t const lds = static_cast<size_t>(s->res_window) * sizeof(resident::dbl2) + fixed(mixed, s->res_width, nt);
	BFMX_CHECK(allow_lds(reinterpret_cast<const void*>(kernel), lds));
	// (tests cut runs into many launches)
	const char* cut = std::getenv("BFMX_RESIDENT_ITERS");
	int64_t const per_launch = cut && std::atoll(cut) > 0 ? std::atoll(cut) : kPerLaunch;
	int64_t const nslots = G > 1 ? 2 * static_cast<int64_t>(G) * kSlotWords : 0;
	int mode = warm ? 1 : 0;
	cap = (std::min(cap, INT64_MAX - kCheckEvery) + kCheckEvery - 1) / kCheckEvery * kCheckEvery;
	while (true) {
		int64_t const stop = std::min(cap, (mode == 2 ? out->iter : 0) + per_launch);
		std::optional<ClusterLock> lock;
		if (G > 1) {
			lock.emplace(s->device, G);
			k_clear<<<static_cast<int>((2 * n + kBlock - 1) / kBlock), kBlock, 0, st>>>(V, 2 * n, nslots);
		}
		kernel<<<G, nt, lds, st>>>(V, poll_limit(), mode, rtol2, delta2, stop, s->d_scal);
		BFMX_HIP(hipGetLastError());
		BFMX_HIP(hipMemcpyAsync(out, s->d_scal, sizeof(Scalars), hipMemcpyDeviceToHost, st));
		BFMX_HIP(hipStreamSynchronize(st));
		if (G > 1 && out->gave_up) {
			s->res_retry = std::chrono::steady_clock::now() + kRetryAfter;
			return BFMX_OK;
		}
		if (out->done != 0 || out->iter >= cap) {
			*ran = true;
			return BFMX_OK;
		}
		mode = 2;
	}
}

// ------------------------------------------------------------------- MINRES
// Workgroups of 512 threads, whose 256 registers hold nine FP64 blocks beside
// the seven vectors of the recurrences: up to 131,072 nodes.
// Measured, 451 nodes (one workgroup, a ring of 40 x 10 cells, 1,349
// iterations): 53 us an iteration with the recurrences on the host and two
// read-backs, here 2.0 us.

namespace {

constexpr int kMinresThreads = 512;

// What a launch leaves.
struct MinresState {
	MinresRun run;
	int32_t gave_up;
};

template <int W>
__global__ __launch_bounds__(kMinresThreads) void k_resident_minres(View V, uint32_t polls, int fresh, double rtol,
                                                                    int64_t stop, int64_t cap,
                                                                    double* __restrict__ more,
                                                                    MinresRun* __restrict__ run) {
	extern __shared__ __align__(16) double dyn[];
	__shared__ Shared sh;
	if (threadIdx.x == 0) {
		sh.polls = polls;
	}
	MinresRun R;
	if (!fresh) {
		R = *run;
	}
	run_minres<W, kMinresThreads>(V, blockIdx.x, gridDim.x, fresh != 0, rtol, stop, cap, more, sh,
	                              reinterpret_cast<resident::dbl2*>(dyn), R);
	// the other workgroups of the cluster read *run before its first all-gather
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		*run = R;
	}
}

}  // namespace

int resident_minres(bfmx_system* s, double rtol, int64_t cap, MinresResult* out, bool* ran) {
	*ran = false;
	const char* e = std::getenv("BFMX_RESIDENT");
	int64_t const n = s->n_nodes, G = (n + kMinresThreads - 1) / kMinresThreads;
	bool const off = (e && e[0] == '0') || std::chrono::steady_clock::now() < s->res_retry;
	int const win = off || G > compute_units(s->device) ? 0 : window_of(s, G, kMinresThreads);
	if (win == 0) {
		return BFMX_OK;
	}
	hipStream_t const st = s->stream;
	double* more = nullptr;       // w and w2 of a run cut at its limit
	MinresState* d_run = nullptr;
	MinresState last{};
	MinresRun& R = last.run;
	bool gave_up = false;
	int const rc = [&]() -> int {
		BFMX_CHECK(palloc(&more, 4 * static_cast<size_t>(n)));
		BFMX_CHECK(palloc(&d_run, 1));
		auto words = [](double* p) { return reinterpret_cast<u64*>(p); };
		View V{s->d_slice_ptr, s->d_col, s->d_diag_blk, s->d_val, nullptr, s->d_bsolve, s->d_x,
		       {words(s->d_r), words(s->d_z), words(s->d_q), words(s->d_p[0])}, words(s->d_p[1]), s->d_dinv,
		       &d_run->gave_up, n};
		int const width = *std::max_element(s->row_len.begin(), s->row_len.end());
		auto const kernel = width <= 7 ? k_resident_minres<7> : k_resident_minres<9>;
		size_t const lds = static_cast<size_t>(win) * sizeof(resident::dbl2);
		BFMX_CHECK(allow_lds(reinterpret_cast<const void*>(kernel), lds));
		const char* cut = std::getenv("BFMX_RESIDENT_ITERS");
		int64_t const per_launch = cut && std::atoll(cut) > 0 ? std::atoll(cut) : kPerLaunch;
		for (int fresh = 1; !gave_up && R.status == 0 && (fresh || R.iter < cap); fresh = 0) {
			int64_t const stop = std::min(cap, R.iter + per_launch);
			std::optional<ClusterLock> lock;
			if (G > 1) {
				lock.emplace(s->device, G);
				k_clear<<<static_cast<int>((2 * n + kBlock - 1) / kBlock), kBlock, 0, st>>>(V, 2 * n,
				                                                                         2 * G * kSlotWords);
			}
			kernel<<<static_cast<unsigned>(G), kMinresThreads, lds, st>>>(V, poll_limit(), fresh, rtol, stop, cap, more,
			                                                              &d_run->run);
			BFMX_HIP(hipGetLastError());
			BFMX_HIP(hipMemcpyAsync(&last, d_run, sizeof last, hipMemcpyDeviceToHost, st));
			BFMX_HIP(hipStreamSynchronize(st));
			gave_up = G > 1 && last.gave_up;
			if (gave_up) {
				s->res_retry = std::chrono::steady_clock::now() + kRetryAfter;
			}
		}
		return BFMX_OK;
	}();
	(void) hipStreamSynchronize(st);   // the block cache takes back drained blocks only
	pfree(more);
	pfree(d_run);
	BFMX_CHECK(rc);
	*ran = !gave_up;
	*out = MinresResult{R.status, R.iter, R.rr, R.bb, R.checks};
	return BFMX_OK;
}

// ------------------------------------------------------------------ batches
// One launch runs many clusters. The systems are sorted into queues by the
// size of the cluster they need; a queue's clusters take its systems largest
// first, one after another. The workgroups (one a CU) are dealt to the queues
// so that they are expected to end together, and neighbouring cluster sizes
// share a launch where that ends sooner. A batch is then bound by the sum of
// its work: in the streaming kernel, one workgroup a system, the largest one's
// time on one CU is the least a launch can take.
// Measured, whole launch with the assembly, block Jacobi to 1e-8: 256 panels of
// 500 to 4,000 nodes 63.2 -> 14.5 ms, 64 panels of 3,000 to 30,000 nodes 835 ->
// 70 ms, 512 of 500 to 30,000 1,911 -> 456 ms.

namespace resident {
namespace {

struct Queue {
	int32_t begin, end;   // in the order of the plan
	int32_t next;
	int32_t pad;
};
struct Member {
	int32_t queue, cluster, g, G;
};

constexpr double kLaunchUs = 20;   // of one launch of clusters
constexpr int kClearParts = 8;   // workgroups clearing one system's words

// Clears what the runs of the plan's systems exchange.
__global__ __launch_bounds__(kBlock) void k_clear_batch(const View* __restrict__ views,
                                                        const int32_t* __restrict__ order,
                                                        const int32_t* __restrict__ groups,
                                                        Queue* __restrict__ queues, int nq, u64* __restrict__ post,
                                                        int npost, Out* __restrict__ out, int nout) {
	int const k = blockIdx.x / kClearParts, part = blockIdx.x % kClearParts;
	int const gid = part * kBlock + threadIdx.x, step = kClearParts * kBlock;
	if (k == 0) {
		for (int i = gid; i < nq; i += step) {
			queues[i].next = queues[i].begin;
		}
		for (int i = gid; i < npost; i += step) {
			post[i] = 0;
		}
		for (int i = gid; i < nout; i += step) {
			out[i].gave_up = 0;
		}
	}
	int const G = groups[k];
	if (G == 1) {
		return;
	}
	View const V = views[order[k]];
	for (int64_t i = gid; i < 2 * V.n; i += step) {
		V.w[0][i] = V.w[1][i] = V.w[2][i] = V.w[3][i] = 0;
	}
	for (int i = gid; i < 2 * G * kSlotWords; i += step) {
		V.slots[i] = 0;
	}
}

template <int W, int PRE>
__global__ __launch_bounds__(kRows) void k_resident_batch(const View* __restrict__ views,
                                                          const int32_t* __restrict__ order,
                                                          const Member* __restrict__ members,
                                                          Queue* __restrict__ queues, u64* __restrict__ post,
                                                          uint32_t polls, double rtol2, int64_t max_iter,
                                                          Out* __restrict__ out) {
	extern __shared__ __align__(16) double dyn[];
	__shared__ Shared sh;
	__shared__ int job;
	if (threadIdx.x == 0) {
		sh.polls = polls;
	}
	Member const M = members[blockIdx.x];
	for (uint32_t round = 1;; round++) {
		if (threadIdx.x == 0) {
			// the cluster's first workgroup takes the next system and posts it
			int k = -1;
			u64* const at = post + M.cluster;
			if (M.g == 0) {
				k = atomicAdd(&queues[M.queue].next, 1);
				k = k < queues[M.queue].end ? order[k] : -1;
				if (M.G > 1) {
					put(at, (static_cast<u64>(static_cast<uint32_t>(k)) << 32) | round);
				}
			} else {
				for (uint32_t spin = 0; spin < sh.polls; spin++) {
					u64 const v = get(at);
					if (static_cast<uint32_t>(v) == round) {
						k = static_cast<int>(v >> 32);
						break;
					}
				}
			}
			job = k;
		}
		__syncthreads();
		int const k = __builtin_amdgcn_readfirstlane(job);
		if (k < 0) {
			break;
		}
		View const V = views[k];
		Run R;
		run_pcg<double, W, PRE, kRows, true>(V, M.g, M.G, 0, rtol2, 0.0, max_iter, true, sh,
		                               reinterpret_cast<resident::dbl2*>(dyn), R);
		if (M.g == 0 && threadIdx.x == 0) {
			out[k].iter = R.iter;
			out[k].rr_true = R.rr_true;
			out[k].bb = R.bb;
			out[k].status = R.status;
			out[k].checks = R.checks;
		}
		if (R.status == kFailed) {
			break;
		}
		__syncthreads();
	}
}

// Sizes of a cluster: the smallest that holds a system's rows is taken.
constexpr int kGroups[] = {1,  2,  3,  4,  5,  6,  7,  8,  10, 12,  14,  16,  18,  20,
                           24, 28, 32, 40, 48, 56, 64, 80, 96, 128, 160, 192, 224, 256};

// Expected microseconds of a system's run: the iterations grow as the square
// root of the nodes (panels of the batched workload: 20 sqrt(n) for 500 to
// 30,000 nodes), an iteration with G workgroups takes what resident.h states.
double run_us(int64_t n, int G) {
	double const it = G == 1 ? 2.5 : G <= 8 ? 5.2 : G <= 64 ? 5.8 : 10.0;
	return 20.0 * std::sqrt(static_cast<double>(n)) * it;
}

// The systems that take clusters of G workgroups.
struct Class {
	int G;
	std::vector<int32_t> members;   // largest first
	double total = 0, longest = 0;  // expected microseconds
	int clusters = 0;

	// when the last of them ends, with c clusters taking them largest first
	double makespan(int c) const {
		double const mean = total / static_cast<double>(members.size());
		return std::max(longest, total / c + (c > 1 ? 0.5 * mean : 0.0));
	}
};

// Clusters of the classes [c0, c1) in one launch of at most cus workgroups:
// one each, then one more wherever the launch ends last, while there is room.
// Returns the launch's expected time (negative: they do not fit).
double share(std::vector<Class>& classes, size_t c0, size_t c1, int cus) {
	int used = 0;
	for (size_t c = c0; c < c1; c++) {
		classes[c].clusters = 1;
		used += classes[c].G;
	}
	if (used > cus) {
		return -1;
	}
	while (true) {
		Class* last = nullptr;
		double worst = 0;
		for (size_t c = c0; c < c1; c++) {
			double const t = classes[c].makespan(classes[c].clusters);
			if (t > worst) {
				worst = t;
				last = &classes[c];
			}
		}
		if (used + last->G > cus || last->clusters == static_cast<int>(last->members.size())) {
			return worst;
		}
		last->clusters++;
		used += last->G;
	}
}

}  // namespace

struct Plan {
	struct Launch {
		int first, blocks;   // its members
	};
	std::vector<Launch> launches;
	std::vector<int32_t> rest;
	int taken = 0, queues = 0, clusters = 0, width = 0;
	int workgroups = 0;   // of the largest launch
	size_t lds = 0;
	View* d_views = nullptr;
	int32_t* d_order = nullptr;
	int32_t* d_groups = nullptr;   // cluster size of each system, in that order
	Member* d_members = nullptr;
	Queue* d_queues = nullptr;
	u64* d_post = nullptr;
};

void plan_destroy(Plan* p) {
	if (!p) {
		return;
	}
	dfree(p->d_views);
	dfree(p->d_order);
	dfree(p->d_groups);
	dfree(p->d_members);
	dfree(p->d_queues);
	dfree(p->d_post);
	delete p;
}

const std::vector<int32_t>& plan_rest(const Plan* p) {
	return p->rest;
}

int plan_workgroups(const Plan* p) {
	return p->workgroups;
}

int plan_create(Plan** out, const std::vector<bfmx_system*>& systems, const std::vector<View>& views,
                hipStream_t st) {
	*out = nullptr;
	int dev = 0;
	BFMX_HIP(hipGetDevice(&dev));
	int const cus = compute_units(dev);
	std::vector<int32_t> by_size(systems.size());
	for (size_t k = 0; k < by_size.size(); k++) {
		by_size[k] = static_cast<int32_t>(k);
	}
	std::stable_sort(by_size.begin(), by_size.end(),
	                 [&](int32_t a, int32_t c) { return systems[a]->n_nodes > systems[c]->n_nodes; });
	std::vector<Class> classes;
	auto* p = new Plan();
	int widest = 0;
	for (int32_t const k : by_size) {
		bfmx_system const* s = systems[k];
		int64_t const need = (s->n_nodes + kRows - 1) / kRows;
		auto const g = std::find_if(std::begin(kGroups), std::end(kGroups), [&](int x) { return x >= need; });
		int const win = g != std::end(kGroups) && *g <= cus ? window_of(s, *g) : 0;
		if (win == 0) {
			p->rest.push_back(k);
			continue;
		}
		if (classes.empty() || classes.back().G != *g) {
			classes.push_back(Class{*g, {}});
		}
		double const us = run_us(s->n_nodes, *g);
		classes.back().members.push_back(k);
		classes.back().total += us;
		classes.back().longest = std::max(classes.back().longest, us);
		widest = std::max(widest, win);
		p->width = std::max(p->width, *std::max_element(s->row_len.begin(), s->row_len.end()));
		p->taken++;
	}
	if (p->taken == 0) {
		delete p;
		return BFMX_OK;
	}
	p->lds = static_cast<size_t>(widest) * sizeof(resident::dbl2) + static_cast<size_t>(fixed(false, p->width, kRows));
	std::vector<int32_t> order, groups;
	std::vector<Queue> queues;
	std::vector<Member> members;
	// neighbouring classes share a launch where that ends sooner than one
	// launch after another: best[c] is the least expected time of the classes
	// from c on, upto[c] the end of their first launch
	size_t const nc = classes.size();
	std::vector<double> best(nc + 1, 0);
	std::vector<size_t> upto(nc + 1, nc);
	for (size_t c0 = nc; c0-- > 0;) {
		best[c0] = -1;
		for (size_t c1 = c0 + 1; c1 <= nc; c1++) {
			double const t = share(classes, c0, c1, cus);
			if (t >= 0 && (best[c0] < 0 || t + kLaunchUs + best[c1] < best[c0])) {
				best[c0] = t + kLaunchUs + best[c1];
				upto[c0] = c1;
			}
		}
	}
	for (size_t c0 = 0; c0 < nc; c0 = upto[c0]) {
		size_t const c1 = upto[c0];
		share(classes, c0, c1, cus);
		int const first = static_cast<int>(members.size());
		for (size_t c = c0; c < c1; c++) {
			Class& C = classes[c];
			int const begin = static_cast<int>(order.size());
			order.insert(order.end(), C.members.begin(), C.members.end());
			groups.insert(groups.end(), C.members.size(), C.G);
			for (int k = 0; k < C.clusters; k++) {
				for (int g = 0; g < C.G; g++) {
					members.push_back(Member{static_cast<int32_t>(queues.size()), p->clusters, g, C.G});
				}
				p->clusters++;
			}
			queues.push_back(Queue{begin, static_cast<int32_t>(order.size()), begin, 0});
		}
		int const blocks = static_cast<int>(members.size()) - first;
		p->launches.push_back(Plan::Launch{first, blocks});
		p->workgroups = std::max(p->workgroups, blocks);
	}
	p->queues = static_cast<int>(queues.size());
	int const rc = [&]() -> int {
		BFMX_CHECK(dalloc(&p->d_views, views.size()));
		BFMX_CHECK(dalloc(&p->d_order, order.size()));
		BFMX_CHECK(dalloc(&p->d_groups, groups.size()));
		BFMX_CHECK(dalloc(&p->d_members, members.size()));
		BFMX_CHECK(dalloc(&p->d_queues, queues.size()));
		BFMX_CHECK(dalloc(&p->d_post, static_cast<size_t>(p->clusters)));
		BFMX_HIP(hipMemcpyAsync(p->d_views, views.data(), views.size() * sizeof(View), hipMemcpyHostToDevice, st));
		BFMX_HIP(hipMemcpyAsync(p->d_order, order.data(), order.size() * sizeof(int32_t), hipMemcpyHostToDevice, st));
		BFMX_HIP(hipMemcpyAsync(p->d_groups, groups.data(), groups.size() * sizeof(int32_t), hipMemcpyHostToDevice,
		                        st));
		BFMX_HIP(hipMemcpyAsync(p->d_members, members.data(), members.size() * sizeof(Member), hipMemcpyHostToDevice,
		                        st));
		BFMX_HIP(hipMemcpyAsync(p->d_queues, queues.data(), queues.size() * sizeof(Queue), hipMemcpyHostToDevice,
		                        st));
		BFMX_HIP(hipStreamSynchronize(st));
		return BFMX_OK;
	}();
	if (rc != BFMX_OK) {
		plan_destroy(p);
		return rc;
	}
	*out = p;
	return BFMX_OK;
}

int plan_launch(Plan* p, hipStream_t st, int precond, double rtol2, int64_t max_iter, Out* d_out, int n) {
	bool const point = precond == BFMX_PRECOND_JACOBI;
	auto const kernel = p->width <= 7
	                        ? (point ? k_resident_batch<7, BFMX_PRECOND_JACOBI> : k_resident_batch<7, BFMX_PRECOND_BLOCK_JACOBI>)
	                        : (point ? k_resident_batch<9, BFMX_PRECOND_JACOBI> : k_resident_batch<9, BFMX_PRECOND_BLOCK_JACOBI>);
	BFMX_CHECK(allow_lds(reinterpret_cast<const void*>(kernel), p->lds));
	k_clear_batch<<<p->taken * kClearParts, kBlock, 0, st>>>(p->d_views, p->d_order, p->d_groups, p->d_queues, p->queues,
	                                                         p->d_post, p->clusters, d_out, n);
	BFMX_HIP(hipGetLastError());
	for (auto const& L : p->launches) {
		kernel<<<L.blocks, kRows, p->lds, st>>>(p->d_views, p->d_order, p->d_members + L.first, p->d_queues, p->d_post,
		                                        poll_limit(), rtol2, max_iter, d_out);
		BFMX_HIP(hipGetLastError());
	}
	return BFMX_OK;
}

}  // namespace resident

}  // namespace bfmx
