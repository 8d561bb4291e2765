// PCG with the matrix held in registers (device code shared by the solve of
// one system and by batches).
//
// The streaming kernels of pcg.hip read the whole matrix from memory in every
// iteration and end each of its two dot products at a kernel boundary: below
// some 260,000 nodes an iteration is then bound by four launches and by the
// latency of its loads, not by bandwidth (13 us an iteration from 451 to
// 23,000 nodes, 32 us at 251,000). Here a cluster of G workgroups runs the
// whole iteration loop in one launch:
//   * one block row per thread, its blocks in registers (a CU's 512 KB of
//     registers hold 1024 rows of nine FP64 blocks), x, r, z and the inverse
//     diagonal beside them;
//   * the direction p of a workgroup's own rows and of the nodes their columns
//     reach (a contiguous window, since the nodes are in RCM order) in LDS;
//     every workgroup forms p = z + beta p for its whole window, so that only
//     z is exchanged;
//   * z and the partial dot products travel through memory in 8-byte words of
//     32 data bits and the 32-bit number of the exchange (the low-latency protocol
//     of collective libraries), written and read with
//     agent-scope relaxed atomics (which pass by the XCDs' incoherent L2s). A
//     reader polls the word itself until it carries the expected number, so an
//     exchange costs one store-to-load latency (1.3 us up to 4 workgroups, 1.8
//     at 32, 2.7 at 256) and needs no fence, no flag and no wait for the stores.
// Measured on one MI355X, microseconds an iteration, streaming -> here: 451 nodes
// (one workgroup) 13.8 -> 1.7; 1,105 (two) 13.4 -> 4.3; 5,124 (six) 13.3 -> 4.6;
// 22,952 (23) 13.4 -> 4.7; 63,126 (62) 16.2 -> 5.0; 251,251 (246) 32.7 -> 10.0,
// point Jacobi on Q1 beams (22,952: block Jacobi, FP32 matrix, P1). Above one
// workgroup the two all-gathers bound it.
// A word is overwritten two exchanges later at the earliest, after an
// all-gather to which every workgroup contributed past its last read of it.
// Every workgroup forms the same sums in the same order, so all of them take
// the same branches; the result does not depend on scheduling.
//
// The workgroups of a cluster must be resident together. A launch has at most
// one workgroup a CU, kernels on other streams end and leave their CUs to it,
// and clusters that could wait for each other's CUs do not run at once: a host
// thread holds a ClusterLock for their CUs (cu_budget.h) from their launch to
// their end (an ordinary launch under the lock costs 11 us with its
// synchronization, a cooperative one 20 us). Between processes nothing prevents that, so every
// wait is bounded (kSpinLimit polls): each workgroup ends whatever happens. A
// vector's node that did not arrive counts as NaN, so that the sums end the run
// in every workgroup; a workgroup whose wait ran out raises the launch's gave_up
// flag, and the host then drops the run, whatever it reports, and solves with the
// streaming kernels.
#pragma once

#include <chrono>

#include "cu_budget.h"
#include "internal.h"

namespace bfmx {

// s - a x accumulated without losing its rounding errors: s carries the
// running sum and c the sum of the errors, so that s + c is the row's
// b - sum A_ij x_j as accurately as if it were summed in twice the working
// precision and then rounded (the product's error exactly from an FMA,
// Knuth's TwoSum for the difference; Ogita, Rump and Oishi, SIAM J. Sci.
// Comput. 26 (2005) 1955-1988, Algorithm Dot2). Contraction is off here: a
// fused s - a x would not be the rounded difference the error terms assume.
__device__ __forceinline__ void sub_exact(double& s, double& c, double a, double x) {
#pragma clang fp contract(off)
	double const p = a * x;
	double const pe = fma(a, x, -p);   // a x = p + pe exactly
	double const t = s - p;
	double const z = t - s;
	double const e = (s - (t - z)) + (-p - z);   // s - p = t + e exactly
	s = t;
	c += e - pe;
}

namespace resident {

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef float flt2 __attribute__((ext_vector_type(2)));
typedef unsigned long long u64;

constexpr uint32_t kSpinLimit = 1u << 22;   // polls of one wait (seconds)
constexpr int kSlotWords = 16;              // a 128-byte line for each workgroup's contribution to an all-gather
                                            // (several in a line cost 0.4 us more at 32 workgroups)
constexpr int kMaxGroup = 256;              // workgroups of a cluster
constexpr int kMaxWindow = 2900;            // nodes of a window (46 KB of the CU's 160 KB of LDS, beside 112 KB)
constexpr int kMaxWidth = 9;                // blocks of a row held in registers
constexpr int kCheckEvery = 16;             // iterations between true-residual checks once one has failed
constexpr int kStall = 8;                   // such checks without halving before the run counts as stalled
constexpr int kFailed = 5;                  // status: a bounded wait ran out
// A wait runs out after seconds, when something else holds the GPU's CUs: the
// system's or batch's solves of the next minute stream without trying again.
constexpr std::chrono::seconds kRetryAfter{60};

// One system's arrays. The exchange uses the solver's vector buffers (16
// bytes a node each): words 0 and 1, 2 and 3 of the two parities in w[0..3],
// the all-gather slots in slots. All five are zeroed before the launch.
struct View {
	const int32_t* slice_ptr;
	const int32_t* col;
	const int32_t* diag_blk;
	const double* val;      // FP64 matrix
	const float* val32;     // FP32 copy (mixed precision)
	const double* b;
	double* x;
	u64* w[4];
	u64* slots;
	double* save;           // 4 doubles a node: r and p of a run cut at its iteration limit
	int32_t* gave_up;       // set by a workgroup whose wait ran out; zeroed before the launch
	int64_t n;
};

// Scalars of a run, the same in every workgroup.
struct Run {
	double rz, rr, bb, tol2, beta, rr_true, rr_ref, rr_best, pq;
	int64_t iter;
	int32_t status;    // 0 running (limit reached), 1 converged, 2 breakdown, 3 stalled, kFailed
	int32_t stall, checking, updates, checks;
};

__device__ __forceinline__ dbl2 ld2(const double* p) {
	return *reinterpret_cast<const dbl2*>(p);
}
__device__ __forceinline__ void st2(double* p, dbl2 v) {
	*reinterpret_cast<dbl2*>(p) = v;
}
__device__ __forceinline__ void put(u64* p, u64 v) {
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get(const u64* p) {
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 word_hi(double v, uint32_t ep) {
	return (static_cast<u64>(__double_as_longlong(v)) & 0xffffffff00000000ull) | ep;
}
__device__ __forceinline__ u64 word_lo(double v, uint32_t ep) {
	return (static_cast<u64>(__double_as_longlong(v)) << 32) | ep;
}
__device__ __forceinline__ double join(u64 hi, u64 lo) {
	return __longlong_as_double(static_cast<long long>((hi & 0xffffffff00000000ull) | (lo >> 32)));
}

template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
	int const lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
	int const hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
	return __hiloint2double(hi, lo);
}

// Sum over each row of 16 lanes, in all of them (register moves between
// lanes: a shuffle through LDS takes several times as long).
__device__ __forceinline__ double row_sum(double v) {
	v += dpp<0xB1>(v);    // lanes 1 0 3 2
	v += dpp<0x4E>(v);    // lanes 2 3 0 1
	v += dpp<0x141>(v);   // the other four of each eight
	v += dpp<0x140>(v);   // the other eight of each sixteen
	return v;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
	return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
	                        __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the wavefront, in all lanes.
__device__ __forceinline__ double wave_total(double v) {
	v = row_sum(v);
	return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// A value that is the same in all lanes, held in scalar registers.
__device__ __forceinline__ double uniform(double v) {
	return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
	                        __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

template <typename MT>
__device__ __forceinline__ const MT* matrix(View const& V) {
	if constexpr (sizeof(MT) == 4) {
		return V.val32;
	} else {
		return V.val;
	}
}

struct Shared {
	double part[3][3][16];   // per kind of all-gather: the waves' partial sums
	double tot[3][3][4];     // the gathered sums of up to four polling waves
	int lo, hi;          // the window
	int below, above;    // own rows before below or from above on lie in another workgroup's window
	int late;            // a wait for a vector's words or the windows ran out
	int failed;          // a wait of an all-gather did: written between the two barriers of gather() only, so
	                     // that all waves read the same after it
	uint32_t polls;      // of one wait at most (set by the kernel; read where a wait goes on)
};

// Blocks of a row held in registers, by threads of the workgroup: six FP64
// blocks (48 registers) fit beside the vectors in the 128 registers a thread
// of 1024 has; the others go to LDS. The loads of the product are kept in order
// (multiply()) and the solution in LDS, or the compiler spills parts of the
// matrix: a spilled register is reloaded through memory in every iteration,
// behind the stores of the exchange (9 us an iteration instead of 4.8).
template <typename MT, int W, int NT>
constexpr int register_blocks() {
	return sizeof(MT) == 8 && NT > 512 && W > 6 ? 6 : W;
}
template <typename MT, int W, int NT>
constexpr int spare_bytes() {
	return (W - register_blocks<MT, W, NT>()) * 4 * static_cast<int>(sizeof(MT)) * NT;
}
// Whether a thread's part of the solution lives in LDS as well (16 bytes each,
// after the spare blocks).
template <typename MT, int NT>
constexpr bool lds_solution() {
	return sizeof(MT) == 8 && NT > 512;
}
template <typename MT, int W, int NT>
constexpr int fixed_bytes() {
	return spare_bytes<MT, W, NT>() + (lds_solution<MT, NT>() ? 16 * NT : 0);
}

// The registers, LDS and exchanges of one workgroup (g of G) of a cluster. MT:
// stored type of the matrix, W: blocks of a row at most, NT: threads.
template <typename MT, int W, int NT>
struct Cluster {
	static constexpr int NW = NT / 64;
	static constexpr int WR = register_blocks<MT, W, NT>();
	typedef MT mt2 __attribute__((ext_vector_type(2)));

	View const& V;
	Shared& sh;
	int const g, G, n;
	int t, lane, wave;
	int r0, r1, row;           // own rows, this thread's
	bool live, shared = false; // it has a row; other workgroups read it
	int lo, nwin, left, own, halo;   // the window: its first node, nodes, nodes before the own rows, own rows, others
	mt2* spare;                // the row's last W - WR blocks, two halves each
	dbl2* win;                 // the vector the matrix is applied to, over the window
	MT m[WR][4];               // the row's first blocks
	uint32_t at[(W + 1) / 2];  // its columns, as places in the window, two a word
	uint32_t ep = 0, sep = 0;  // exchanges of a vector and all-gathers so far

	__device__ __forceinline__ Cluster(View const& v, Shared& s, int wg, int groups, dbl2* lds)
	    : V(v), sh(s), g(wg), G(groups), n(static_cast<int>(v.n)) {
		spare = reinterpret_cast<mt2*>(lds);
		win = lds + fixed_bytes<MT, W, NT>() / sizeof(dbl2);
		t = threadIdx.x;
		lane = t & 63;
		wave = __builtin_amdgcn_readfirstlane(t >> 6);
		int const rows = ((n + G - 1) / G + 63) / 64 * 64;   // per workgroup (at most NT)
		r0 = min(g * rows, n);
		r1 = min(r0 + rows, n);
		row = r0 + t;
		live = row < r1;
		if (t == 0) {
			sh.lo = r0;
			sh.hi = r1;
			sh.below = 0;
			sh.above = n;
			sh.late = 0;
			sh.failed = 0;
		}
		__syncthreads();
		int clo = r0, chi = r0;
		int const r64 = row & 63;
		int beg = 0, len = 0;   // the row's first block, and blocks (padding included)
		if (live) {
			beg = V.slice_ptr[row >> 6] + r64;
			len = (V.slice_ptr[(row >> 6) + 1] - beg + 63) >> 6;
			clo = chi = row;
		}
#pragma unroll
		for (int k = 0; k < W; k++) {
			mt2 a = {0, 0}, c = {0, 0};
			if (k < len) {
				int64_t const blk = beg + k * kSlice;
				int const col = V.col[blk];
				const MT* const from = matrix<MT>(V) + 4 * blk - 2 * r64;
				a = *reinterpret_cast<const mt2*>(from);
				c = *reinterpret_cast<const mt2*>(from + 2 * kSlice);
				clo = min(clo, col);
				chi = max(chi, col);
			}
			if (k < WR) {
				m[k < WR ? k : 0][0] = a.x;
				m[k < WR ? k : 0][1] = a.y;
				m[k < WR ? k : 0][2] = c.x;
				m[k < WR ? k : 0][3] = c.y;
			} else {
				spare[(2 * (k - WR)) * NT + t] = a;
				spare[(2 * (k - WR) + 1) * NT + t] = c;
			}
			__builtin_amdgcn_sched_barrier(0);   // one block at a time: few registers
		}
		if (live) {
			atomicMin(&sh.lo, clo);
			atomicMax(&sh.hi, chi + 1);
		}
		__syncthreads();
		lo = __builtin_amdgcn_readfirstlane(sh.lo);
		nwin = __builtin_amdgcn_readfirstlane(sh.hi) - lo;
		left = r0 - lo;
		own = r1 - r0;
		halo = nwin - own;
		// A workgroup without rows (a cluster may be larger than its system needs)
		// has no window, yet multiplies its zero blocks by place 0: what was left
		// there may be a NaN. Read behind the barriers of the caller's first steps.
		if (nwin == 0 && t == 0) {
			win[0] = dbl2{0, 0};
		}
		// a block past the row's end (its values are zero) takes place 0
		auto place = [&](int k) { return k < len ? static_cast<uint32_t>(V.col[beg + k * kSlice] - lo) : 0u; };
#pragma unroll
		for (int k = 0; k < W; k += 2) {
			at[k / 2] = place(k) | (k + 1 < W ? place(k + 1) << 16 : 0u);
			__builtin_amdgcn_sched_barrier(0);
		}
		if (G > 1) {
			share_windows();
		}
	}

	// The rows that other workgroups read: the first all-gather is of the
	// windows.
	__device__ __forceinline__ void share_windows() {
		sep = 1;
		u64* const base = V.slots + static_cast<int64_t>(G) * kSlotWords;
		if (t < 2) {
			put(base + g * kSlotWords + t, (static_cast<u64>(t == 0 ? lo : lo + nwin) << 32) | sep);
		}
		if (t < G && t != g) {
			u64 a, c;
			uint32_t spin = 0;
#pragma unroll 1
			while (true) {
				a = get(base + t * kSlotWords);
				c = get(base + t * kSlotWords + 1);
				if (static_cast<uint32_t>(a) == sep && static_cast<uint32_t>(c) == sep) {
					break;
				}
				if (++spin >= sh.polls) {
					sh.late = 1;
					break;
				}
			}
			if (t < g) {
				atomicMax(&sh.below, static_cast<int>(c >> 32));
			} else {
				atomicMin(&sh.above, static_cast<int>(a >> 32));
			}
		}
		__syncthreads();
		shared = live && (row < sh.below || row >= sh.above);
	}

	// The diagonal block of the own row.
	__device__ __forceinline__ void diagonal(double& a00, double& a01, double& a10, double& a11) const {
		const double* top = V.val + 4 * static_cast<int64_t>(V.diag_blk[row]) - 2 * (row & 63);
		a00 = top[0];
		a01 = top[1];
		a10 = top[2 * kSlice];
		a11 = top[2 * kSlice + 1];
	}

	// At the end of a run. A gather after the last wait made the flags visible,
	// but for waits at an iteration limit whose values are not used any more.
	__device__ __forceinline__ void report() const {
		if (t == 0 && (sh.late || sh.failed)) {
			*V.gave_up = 1;
		}
	}

	// Addresses are formed anew in every iteration: held in registers they would
	// push the matrix out.
	__device__ __forceinline__ void forget_addresses() {
		asm volatile("" : "+v"(t), "+v"(row));
	}

	// After a gather.
	__device__ __forceinline__ bool failed() const {
		return __builtin_amdgcn_readfirstlane(sh.failed) != 0;
	}

	// Word k (0 .. 3) of node i in the current exchange (byte offsets below
	// 2^32: a uniform base and one 32-bit register).
	__device__ __forceinline__ u64* word_at(int k, int i) const {
		u64* const base = (ep & 1 ? V.w[2 + k / 2] : V.w[k / 2]) + (k & 1 ? n : 0);
		return reinterpret_cast<u64*>(reinterpret_cast<char*>(base) + static_cast<uint32_t>(i) * 8u);
	}

	__device__ __forceinline__ void publish(dbl2 v) {
		ep++;
		if (shared) {
			put(word_at(0, row), word_hi(v.x, ep));
			put(word_at(1, row), word_lo(v.x, ep));
			put(word_at(2, row), word_hi(v.y, ep));
			put(word_at(3, row), word_lo(v.y, ep));
		}
	}

	// The last published vector at node i of another workgroup.
	__device__ __forceinline__ dbl2 receive(int i) const {
		u64 q0, q1, q2, q3;
		uint32_t spin = 0;
#pragma unroll 1
		while (true) {
			q0 = get(word_at(0, i));
			q1 = get(word_at(1, i));
			q2 = get(word_at(2, i));
			q3 = get(word_at(3, i));
			if (static_cast<uint32_t>(q0) == ep && static_cast<uint32_t>(q1) == ep &&
			    static_cast<uint32_t>(q2) == ep && static_cast<uint32_t>(q3) == ep) {
				break;
			}
			if (++spin >= sh.polls) {
				sh.late = 1;
				q0 = q1 = q2 = q3 = ~u64{0};   // NaN
				break;
			}
		}
		return dbl2{join(q0, q1), join(q2, q3)};
	}

	// Place in the window of its node k without the own rows.
	__device__ __forceinline__ int halo_at(int k) const {
		return k < left ? k : k + own;
	}

	// Sums v over the cluster (the same value everywhere); meanwhile `work` runs
	// between the posting of the contribution and the wait for the others'.
	// set: the LDS arrays used (callers alternate, so that no array is written
	// while a wave may still read it). NV <= 3.
	template <int NV, typename Work>
	__device__ __forceinline__ void gather(double (&v)[NV], int set, Work&& work) {
#pragma unroll
		for (int k = 0; k < NV; k++) {
			double const s = wave_total(v[k]);
			if (lane == 0) {
				sh.part[set][k][wave] = s;
			}
		}
		__syncthreads();
		auto total = [&](int k) { return row_sum((lane & 15) < NW ? sh.part[set][k][lane & 15] : 0.0); };
		if (G == 1) {
#pragma unroll
			for (int k = 0; k < NV; k++) {
				v[k] = uniform(total(k));
			}
			work();
			return;
		}
		sep++;
		u64* const base = V.slots + static_cast<int64_t>(sep & 1) * G * kSlotWords;
		if (wave == 0) {
			double s[NV];
#pragma unroll
			for (int k = 0; k < NV; k++) {
				s[k] = total(k);
			}
#pragma unroll
			for (int k = 0; k < NV; k++) {
				if (lane == 2 * k) {
					put(base + g * kSlotWords + lane, word_hi(s[k], sep));
				}
				if (lane == 2 * k + 1) {
					put(base + g * kSlotWords + lane, word_lo(s[k], sep));
				}
			}
		}
		work();
		if (wave < (G + 63) / 64) {
			u64 q[2 * NV];
#pragma unroll
			for (int k = 0; k < 2 * NV; k++) {
				q[k] = 0;
			}
			if (t < G) {
				const u64* const from = base + t * kSlotWords;
				uint32_t spin = 0;
#pragma unroll 1
				while (true) {
					bool ok = true;
#pragma unroll
					for (int k = 0; k < 2 * NV; k++) {
						q[k] = get(from + k);
					}
#pragma unroll
					for (int k = 0; k < 2 * NV; k++) {
						ok = ok && static_cast<uint32_t>(q[k]) == sep;
					}
					if (ok) {
						break;
					}
					if (++spin >= sh.polls) {
						sh.failed = 1;
						break;
					}
				}
			}
#pragma unroll
			for (int k = 0; k < NV; k++) {
				double const s = wave_total(join(q[2 * k], q[2 * k + 1]));
				if (lane == 0) {
					sh.tot[set][k][wave] = s;
				}
			}
		}
		__syncthreads();
#pragma unroll
		for (int k = 0; k < NV; k++) {
			double s = sh.tot[set][k][0];
			for (int w = 1; w < (G + 63) / 64; w++) {
				s += sh.tot[set][k][w];
			}
			v[k] = uniform(s);
		}
	}
	template <int NV>
	__device__ __forceinline__ void gather(double (&v)[NV], int set) {
		gather(v, set, [] {});
	}

	// The matrix times the window, own row (two accumulators a component).
	__device__ __forceinline__ dbl2 multiply() {
		dbl2 q = {0, 0}, qodd = {0, 0};
#pragma unroll
		for (int k = 0; k < (W + 1) / 2; k++) {
			asm volatile("" : "+v"(at[k]));   // unpacked in every iteration, not held unpacked
		}
#pragma unroll
		for (int k = 0; k < W; k++) {
			dbl2 const pv = win[(at[k / 2] >> (16 * (k & 1))) & 0xffffu];
			mt2 a, c;
			if (k < WR) {
				int const kr = k < WR ? k : 0;
				if constexpr (sizeof(MT) == 4) {
					// converted in every iteration: kept as FP64 they would not fit
					asm volatile("" : "+v"(m[kr][0]), "+v"(m[kr][1]), "+v"(m[kr][2]), "+v"(m[kr][3]));
				}
				a = mt2{m[kr][0], m[kr][1]};
				c = mt2{m[kr][2], m[kr][3]};
			} else {
				a = spare[(2 * (k - WR)) * NT + t];
				c = spare[(2 * (k - WR) + 1) * NT + t];
			}
			dbl2& s = k & 1 ? qodd : q;
			s.x = fma(static_cast<double>(a.x), pv.x, s.x);
			s.x = fma(static_cast<double>(a.y), pv.y, s.x);
			s.y = fma(static_cast<double>(c.x), pv.x, s.y);
			s.y = fma(static_cast<double>(c.y), pv.y, s.y);
			if (NT > 512 && k % 2 == 1) {
				// the next loads wait for these products: the registers hold the matrix
				asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(qodd.x), "+v"(qodd.y)::"memory");
			}
		}
		return q + qodd;
	}

	// b - A x of the own row with the FP64 matrix, compensated (row_residual in
	// pcg.hip). x is published for it; the own rows of the window are left
	// holding keep. HALVES: one half of a block at a time, in fewer registers.
	template <bool HALVES = false>
	__device__ __forceinline__ dbl2 true_residual(dbl2 x, dbl2 keep) {
		publish(x);
		dbl2 res = {0, 0};
		__syncthreads();
		if (live) {
			win[row - lo] = x;
		}
		__syncthreads();
		if (live) {
			dbl2 const bv = ld2(V.b + 2 * static_cast<int64_t>(row));
			int const r64 = row & 63, beg = V.slice_ptr[row >> 6] + r64, end = V.slice_ptr[(row >> 6) + 1];
			double s0 = bv.x, s1 = bv.y, c0 = 0, c1 = 0;
#pragma unroll 1
			for (int blk = beg; blk < end; blk += kSlice) {
				int const c = V.col[blk];
				int64_t const o = 4 * static_cast<int64_t>(blk) - 2 * r64;
				dbl2 const a = ld2(V.val + o);
				dbl2 d = {0, 0};
				if (!HALVES) {
					d = ld2(V.val + o + 2 * kSlice);
				}
				dbl2 const xv = c >= r0 && c < r1 ? win[c - lo] : receive(c);
				sub_exact(s0, c0, a.x, xv.x);
				sub_exact(s0, c0, a.y, xv.y);
				if (HALVES) {
					asm volatile("" : "+v"(s0), "+v"(c0)::"memory");
					d = ld2(V.val + o + 2 * kSlice);
				}
				sub_exact(s1, c1, d.x, xv.x);
				sub_exact(s1, c1, d.y, xv.y);
			}
			res = dbl2{s0 + c0, s1 + c1};
		}
		__syncthreads();
		if (live) {
			win[row - lo] = keep;
		}
		return res;
	}
};

// One PCG run, called by all NT threads of workgroup g of G. On return R holds
// the run's scalars (in every thread) and V.x the solution of the workgroup's
// rows. lds: the spare blocks and the window. mode 0 starts from x = 0, 1 from
// the x in V.x, 2 continues a run cut at its limit (R as it was left, r and p in
// V.save). Runs until R.iter >= stop. A workgroup that left because a wait ran
// out leaves its part of V.x as it was.
// LEAN forms z = M^-1 r again where p needs it instead of keeping it, and takes the
// blocks of a true residual by halves. One system's block Jacobi with 1024 threads
// otherwise spills 12 registers, outside its loop but for one load and store,
// which hide: 915 nodes 2.65 us an iteration, LEAN 2.69; 5,124 4.72 either way;
// 22,857 4.87, LEAN 4.98. There it is for the solve that allocates nothing: for
// the first launch that needs scratch memory the runtime takes some from the
// device (16 MiB). The batch kernels carry more
// state and spill 20 to 27 registers, LEAN 10 to 13, most of them in the true
// residual: 256 panels of 500 to 4,000 nodes 15.7 ms with point and 15.2 with
// block Jacobi, LEAN 14.9 and 14.3; 24 of 10,000 to 30,000 45.9 and 45.5, LEAN
// 42.8 and 41.5.
template <typename MT, int W, int PRE, int NT, bool LEAN = false>
__device__ void run_pcg(View const& V, int g, int G, int mode, double rtol2, double delta2, int64_t stop,
                        bool final_check, Shared& sh, dbl2* lds, Run& R) {
	constexpr int kAhead = 1;   // halo nodes a thread reads while it waits for the sums
	Cluster<MT, W, NT> C(V, sh, g, G, lds);
	dbl2 dinv0 = {0, 0}, dinv1 = {0, 0};
	if (C.live) {
		double a00, a01, a10, a11;
		C.diagonal(a00, a01, a10, a11);
		if (PRE == BFMX_PRECOND_JACOBI) {
			dinv0 = dbl2{1.0 / a00, 1.0 / a11};
		} else {
			double const det = a00 * a11 - a01 * a10;
			dinv0 = dbl2{a11 / det, -a01 / det};
			dinv1 = dbl2{-a10 / det, a00 / det};
		}
	}
	auto precond = [&](dbl2 r) {
		if (PRE == BFMX_PRECOND_JACOBI) {
			return dbl2{dinv0.x * r.x, dinv0.y * r.y};
		}
		return dbl2{dinv0.x * r.x + dinv0.y * r.y, dinv1.x * r.x + dinv1.y * r.y};
	};
	dbl2 r = {0, 0}, z = {0, 0}, pn = {0, 0};
	// the own x: in a register, or in this thread's own place in LDS
	dbl2 xr = {0, 0};
	dbl2* const xs = lds + spare_bytes<MT, W, NT>() / sizeof(dbl2);
	auto x_get = [&]() {
		if constexpr (lds_solution<MT, NT>()) {
			return xs[C.t];
		} else {
			return xr;
		}
	};
	auto x_set = [&](dbl2 v) {
		if constexpr (lds_solution<MT, NT>()) {
			xs[C.t] = v;
		} else {
			xr = v;
		}
	};
	x_set(dbl2{0, 0});
	double beta = 0;
	int status = 0;
	for (int k = C.t; k < C.nwin; k += NT) {
		C.win[k] = mode == 2 ? ld2(V.save + 2 * (static_cast<int64_t>(C.n) + C.lo + k)) : dbl2{0, 0};
	}
	if (mode == 2) {
		if (C.live) {
			x_set(ld2(V.x + 2 * static_cast<int64_t>(C.row)));
			r = ld2(V.save + 2 * static_cast<int64_t>(C.row));
			z = precond(r);
		}
		beta = R.beta;
		__syncthreads();
	} else {
		__syncthreads();
		if (C.live) {
			if (mode == 1) {
				x_set(ld2(V.x + 2 * static_cast<int64_t>(C.row)));
			} else {
				r = ld2(V.b + 2 * static_cast<int64_t>(C.row));
			}
		}
		if (mode == 1) {
			r = C.template true_residual<LEAN>(x_get(), pn);
		}
		z = precond(r);
		dbl2 const bv = C.live ? ld2(V.b + 2 * static_cast<int64_t>(C.row)) : dbl2{0, 0};
		double v[3] = {r.x * z.x + r.y * z.y, r.x * r.x + r.y * r.y, bv.x * bv.x + bv.y * bv.y};
		C.gather(v, 2);
		R.rz = v[0];
		R.rr = R.rr_true = R.rr_ref = v[1];
		R.bb = v[2];
		R.tol2 = uniform(rtol2 * v[2]);
		R.rr_best = R.pq = 0;
		R.iter = 0;
		R.stall = R.checking = R.checks = 0;
		R.updates = 1;
		status = C.failed() ? kFailed : R.rr <= R.tol2 ? 1 : 0;
	}
	if (status == 0 && R.iter < stop) {
		C.publish(z);
	}
	dbl2 hz[kAhead];   // z of this thread's first halo nodes
	auto halo_first = [&] {
#pragma unroll
		for (int u = 0; u < kAhead; u++) {
			int const k = C.t + u * NT;
			if (k < C.halo) {
				hz[u] = C.receive(C.lo + C.halo_at(k));
			}
		}
	};
	if (status == 0 && R.iter < stop) {
		halo_first();
	}
	while (status == 0 && R.iter < stop) {
		C.forget_addresses();
		if (LEAN) {
			asm volatile("" : "+v"(r.x), "+v"(r.y));   // or the compiler keeps z after all
			z = precond(r);
		}
		// p = z + beta p over the window
		if (C.live) {
			pn = z + beta * C.win[C.row - C.lo];
			C.win[C.row - C.lo] = pn;
		}
#pragma unroll
		for (int u = 0; u < kAhead; u++) {
			int const k = C.t + u * NT;
			if (k < C.halo) {
				int const a = C.halo_at(k);
				C.win[a] = hz[u] + beta * C.win[a];
			}
		}
		for (int k = C.t + kAhead * NT; k < C.halo; k += NT) {
			int const a = C.halo_at(k);
			C.win[a] = C.receive(C.lo + a) + beta * C.win[a];
		}
		__syncthreads();
		dbl2 const q = C.multiply();
		double v1[1] = {pn.x * q.x + pn.y * q.y};
		C.gather(v1, 0);
		R.pq = v1[0];
		if (C.failed()) {
			status = kFailed;
			break;
		}
		if (!(v1[0] > 0) || !isfinite(v1[0])) {
			status = 2;
			break;
		}
		double const alpha = uniform(R.rz / v1[0]);
		x_set(x_get() + alpha * pn);
		r -= alpha * q;
		z = precond(r);
		C.publish(z);
		double v2[2] = {r.x * z.x + r.y * z.y, r.x * r.x + r.y * r.y};
		C.gather(v2, 1, halo_first);
		if (C.failed()) {
			status = kFailed;
			break;
		}
		R.iter++;
		double const rz_prev = R.rz;
		beta = uniform(v2[0] / rz_prev);
		R.rz = v2[0];
		R.rr = v2[1];
		bool const at_tol = R.rr <= R.tol2;
		bool const every = R.iter % kCheckEvery == 0;
		if ((at_tol && !R.checking) || (every && (R.checking || R.rr <= delta2 * R.rr_ref))) {
			// the true residual replaces the recursive one (the directions are
			// kept) and decides about the end
			r = C.template true_residual<LEAN>(x_get(), pn);
			z = precond(r);
			double v3[2] = {r.x * z.x + r.y * z.y, r.x * r.x + r.y * r.y};
			C.gather(v3, 2);
			if (C.failed()) {
				status = kFailed;
				break;
			}
			beta = rz_prev != 0 ? uniform(v3[0] / rz_prev) : 0.0;
			R.rz = v3[0];
			R.rr = R.rr_true = R.rr_ref = v3[1];
			R.updates++;
			R.checks++;
			if (R.rr <= R.tol2) {
				status = 1;
			} else {
				if (at_tol || R.checking) {
					R.checking = 1;
					if (R.rr_best == 0 || R.rr < 0.25 * R.rr_best) {
						R.rr_best = R.rr;
						R.stall = 0;
					} else if (++R.stall >= kStall) {
						status = 3;
					}
				}
				if (status == 0) {
					C.publish(z);
					halo_first();
				}
			}
		}
	}
	R.beta = beta;
	if (status == 0 && final_check && R.checks == 0) {
		dbl2 const rt = C.template true_residual<LEAN>(x_get(), pn);
		double v[1] = {rt.x * rt.x + rt.y * rt.y};
		C.gather(v, 2);
		R.rr_true = v[0];
		if (C.failed()) {
			status = kFailed;
		}
	}
	R.status = status;
	C.report();
	if (C.live && status != kFailed) {
		st2(V.x + 2 * static_cast<int64_t>(C.row), x_get());
		if (status == 0) {
			st2(V.save + 2 * static_cast<int64_t>(C.row), r);
			st2(V.save + 2 * (static_cast<int64_t>(C.n) + C.row), pn);
		}
	}
}

// Scalars of a MINRES run, the same in every workgroup (solve_minres in pcg.hip
// names them).
struct MinresRun {
	double oldb, beta, dbar, epsln, phibar, cs, sn, beta1, bb, rr;
	int64_t iter, next_check;
	int32_t status;    // 0 running (limit reached), 1 converged, 2 breakdown, 3 exhausted above rtol, kFailed
	int32_t checks;
};

// MINRES with the matrix in registers, preconditioned by 1 / |diagonal|: the
// recurrences of solve_minres (pcg.hip) on the device, in every thread; two
// all-gathers an iteration where the streaming form has two synchronous
// read-backs. fresh starts from x = 0; else the run goes on from V.x and the
// vectors r1, r2, w, w2 in V.save and more (2 n doubles each). Runs until
// R.iter >= stop; the residual is checked at iteration cap whatever its estimate.
template <int W, int NT>
__device__ void run_minres(View const& V, int g, int G, bool fresh, double rtol, int64_t stop, int64_t cap,
                           double* more, Shared& sh, dbl2* lds, MinresRun& R) {
	Cluster<double, W, NT> C(V, sh, g, G, lds);
	int64_t const n2 = 2 * static_cast<int64_t>(C.n);
	dbl2 dinv = {0, 0};
	dbl2 x = {0, 0}, r1 = {0, 0}, r2 = {0, 0}, y = {0, 0}, w = {0, 0}, w2 = {0, 0};
	if (C.live) {
		double a00, a01, a10, a11;
		C.diagonal(a00, a01, a10, a11);
		dinv = dbl2{a00 != 0 ? 1.0 / fabs(a00) : 1.0, a11 != 0 ? 1.0 / fabs(a11) : 1.0};
		int64_t const i = 2 * static_cast<int64_t>(C.row);
		if (fresh) {
			r1 = r2 = ld2(V.b + i);
		} else {
			x = ld2(V.x + i);
			r1 = ld2(V.save + i);
			r2 = ld2(V.save + n2 + i);
			w = ld2(more + i);
			w2 = ld2(more + n2 + i);
		}
		y = dinv * r2;
	}
	if (fresh) {
		double v[2] = {r2.x * y.x + r2.y * y.y, r2.x * r2.x + r2.y * r2.y};
		C.gather(v, 2);
		R = MinresRun{};
		R.bb = R.rr = v[1];
		R.cs = -1;
		R.beta1 = R.beta = R.phibar = uniform(sqrt(v[0]));
		if (C.failed()) {
			R.status = kFailed;
		} else if (!(v[0] > 0)) {
			R.status = v[1] == 0 ? 1 : 2;   // b = 0: x = 0; else M is not positive
		}
	}
	double const tol2 = uniform(rtol * rtol * R.bb);
	dbl2 hy = {0, 0};   // y of this thread's first halo node
	auto halo_first = [&] {
		if (C.t < C.halo) {
			hy = C.receive(C.lo + C.halo_at(C.t));
		}
	};
	bool const runs = R.status == 0 && R.iter < stop;
	if (runs) {
		C.publish(y);
		halo_first();
	}
	while (R.status == 0 && R.iter < stop) {
		C.forget_addresses();
		if (C.live) {
			C.win[C.row - C.lo] = y;
		}
		if (C.t < C.halo) {
			C.win[C.halo_at(C.t)] = hy;
		}
		for (int k = C.t + NT; k < C.halo; k += NT) {
			int const a = C.halo_at(k);
			C.win[a] = C.receive(C.lo + a);
		}
		__syncthreads();
		int64_t const it = R.iter + 1;
		double const sy = uniform(1.0 / R.beta), sr = it >= 2 ? uniform(R.beta / R.oldb) : 0.0;
		dbl2 const v = sy * y;
		dbl2 yn = sy * C.multiply() - sr * r1;
		double d[1] = {v.x * yn.x + v.y * yn.y};
		C.gather(d, 0);
		double const alfa = d[0];
		yn -= uniform(alfa / R.beta) * r2;
		y = dinv * yn;
		C.publish(y);
		d[0] = yn.x * y.x + yn.y * y.y;
		C.gather(d, 1, halo_first);
		if (C.failed()) {
			R.status = kFailed;
			break;
		}
		R.iter = it;
		if (!(d[0] >= 0) || !isfinite(alfa)) {
			R.status = 2;   // the preconditioner is not positive definite, or overflow
			break;
		}
		r1 = r2;
		r2 = yn;
		R.oldb = R.beta;
		R.beta = uniform(sqrt(d[0]));
		double const oldeps = R.epsln;
		double const delta = uniform(R.cs * R.dbar + R.sn * alfa);
		double const gbar = uniform(R.sn * R.dbar - R.cs * alfa);
		R.epsln = uniform(R.sn * R.beta);
		R.dbar = uniform(-R.cs * R.beta);
		double const gamma = uniform(fmax(hypot(gbar, R.beta), 1e-300));
		R.cs = uniform(gbar / gamma);
		R.sn = uniform(R.beta / gamma);
		double const phi = uniform(R.cs * R.phibar);
		R.phibar = uniform(R.sn * R.phibar);
		// w_new = (v - oldeps w2 - delta w) / gamma; (w2, w) <- (w, w_new)
		double const rgamma = uniform(1.0 / gamma);
		dbl2 const wn = (v - oldeps * w2 - delta * w) * rgamma;
		w2 = w;
		w = wn;
		x += phi * wn;
		// the M^-1-norm estimate phibar triggers a true residual check
		if ((R.phibar <= rtol * R.beta1 && it >= R.next_check) || R.beta == 0 || it == cap) {
			dbl2 const res = C.true_residual(x, y);
			d[0] = res.x * res.x + res.y * res.y;
			C.gather(d, 2);
			if (C.failed()) {
				R.status = kFailed;
				break;
			}
			R.rr = d[0];
			R.checks++;
			R.next_check = it + 10;
			if (d[0] <= tol2) {
				R.status = 1;
			} else if (R.beta == 0) {
				R.status = 3;   // the Krylov space is exhausted above rtol
			} else {
				C.publish(y);
				halo_first();
			}
		}
	}
	C.report();
	if (C.live && R.status != kFailed) {
		int64_t const i = 2 * static_cast<int64_t>(C.row);
		st2(V.x + i, x);
		if (R.status == 0) {
			st2(V.save + i, r1);
			st2(V.save + n2 + i, r2);
			st2(more + i, w);
			st2(more + n2 + i, w2);
		}
	}
}

// Most block rows of a workgroup, one per thread.
constexpr int kRows = 1024;

// Compute units of a device: the most workgroups of a launch of clusters.
int compute_units(int device);

// Held by a thread from its launch of `workgroups` workgroups in clusters until
// they have ended (its stream drained).
class ClusterLock {
public:
	ClusterLock(int device, int64_t workgroups);
	~ClusterLock();
	ClusterLock(ClusterLock const&) = delete;
	ClusterLock& operator=(ClusterLock const&) = delete;

private:
	CuBudget& m_budget;
	int const m_share;
};

// The nodes of the widest window when G workgroups of at most `threads` rows
// share the system's (0: they cannot, or a window or row is too long for the
// kernels above).
int window_of(const bfmx_system* s, int64_t G, int threads = kRows);

// ---- batches (resident.hip)

// What a system's run of a batch reports.
struct Out {
	int64_t iter;
	double rr_true;
	double bb;
	int32_t status;   // 1 converged, 2 breakdown, 3 stagnated, 0 iteration limit, kFailed
	int32_t checks;
	int32_t gave_up;  // a workgroup's wait ran out: the rest does not count
};

struct Plan;
// The clusters for a batch of systems (views[k]: system k's arrays; they must
// stay). *out is null when no system fits.
int plan_create(Plan** out, const std::vector<bfmx_system*>& systems, const std::vector<View>& views,
                hipStream_t st);
void plan_destroy(Plan* p);
// Systems the plan does not take, largest first.
const std::vector<int32_t>& plan_rest(const Plan* p);
// Workgroups of the plan's largest launch.
int plan_workgroups(const Plan* p);
// Queues the runs of the plan's systems (the caller holds a ClusterLock for
// plan_workgroups until st is drained). If any of the n systems of d_out has gave_up set afterwards,
// some of the plan's were not solved.
int plan_launch(Plan* p, hipStream_t st, int precond, double rtol2, int64_t max_iter, Out* d_out, int n);

}  // namespace resident
}  // namespace bfmx
