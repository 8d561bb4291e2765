// Host side of the register-resident PCG (resident.h): which systems it takes,
// its launches for one system, and the fall-back to the streaming kernels.

#include <algorithm>
#include <cstdlib>

#include "resident.h"

namespace bfmx {

using namespace resident;

namespace {

constexpr int kRows = 1024;             // block rows of a workgroup, one per thread
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
}

template <typename MT, int W, int PRE, int NT>
__global__ __launch_bounds__(NT) void k_resident_pcg(View V, int mode, double rtol2, double delta2, int64_t stop,
                                                     Scalars* __restrict__ S) {
	extern __shared__ double dyn[];
	__shared__ Shared sh;
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
	run_pcg<MT, W, PRE, NT>(V, blockIdx.x, gridDim.x, mode, rtol2, delta2, stop, false, sh,
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

typedef void (*PcgKernel)(View, int, double, double, int64_t, Scalars*);

template <typename MT, int W, int PRE>
PcgKernel pick_threads(int nt) {
	return nt == 512 ? k_resident_pcg<MT, W, PRE, 512> : k_resident_pcg<MT, W, PRE, 1024>;
}

template <typename MT, int W>
PcgKernel pick_precond(int pre, int nt) {
	return pre == BFMX_PRECOND_JACOBI ? pick_threads<MT, W, BFMX_PRECOND_JACOBI>(nt)
	                                  : pick_threads<MT, W, BFMX_PRECOND_BLOCK_JACOBI>(nt);
}

PcgKernel pick(bool mixed, int width, int pre, int nt) {
	if (mixed) {
		return width <= 7 ? pick_precond<float, 7>(pre, nt) : pick_precond<float, 9>(pre, nt);
	}
	return width <= 7 ? pick_precond<double, 7>(pre, nt) : pick_precond<double, 9>(pre, nt);
}

// LDS bytes of the row blocks that do not fit the registers.
int spare(bool mixed, int width, int nt) {
	return mixed || nt <= 512 ? 0 : width <= 7 ? spare_bytes<double, 7, 1024>() : spare_bytes<double, 9, 1024>();
}

}  // namespace

namespace resident {

bool fits(const bfmx_system* s, int* groups, int* window) {
	int64_t const n = s->n_nodes;
	int64_t const G = (n + kRows - 1) / kRows;
	if (n == 0 || G > kMaxGroup) {
		return false;
	}
	if (*std::max_element(s->row_len.begin(), s->row_len.end()) > kMaxWidth) {
		return false;
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
	*groups = static_cast<int>(G);
	*window = widest;
	return widest <= kMaxWindow;
}

}  // namespace resident

int resident_pcg(bfmx_system* s, int precond, bool mixed, double rtol2, double delta2, int64_t cap, bool warm,
                 Scalars* out, bool* ran) {
	*ran = false;
	const char* e = std::getenv("BFMX_RESIDENT");
	if ((e && e[0] == '0') || s->n_conv_seg > 0 || (precond != BFMX_PRECOND_JACOBI && precond != BFMX_PRECOND_BLOCK_JACOBI)) {
		return BFMX_OK;
	}
	if (s->res_groups < 0) {
		int G = 0, win = 0;
		s->res_groups = fits(s, &G, &win) ? G : 0;
		s->res_window = win;
		s->res_width = *std::max_element(s->row_len.begin(), s->row_len.end());
	}
	int const G = s->res_groups;
	if (G == 0) {
		return BFMX_OK;
	}
	hipStream_t const st = s->stream;
	int64_t const n = s->n_nodes;
	auto words = [](double* p) { return reinterpret_cast<u64*>(p); };
	View V{s->d_slice_ptr, s->d_col, s->d_diag_blk, s->d_val, s->d_val32, s->d_bsolve, s->d_x,
	       {words(s->d_r), words(s->d_z), words(s->d_q), words(s->d_p[0])}, words(s->d_p[1]), s->d_dinv, n};
	int const nt = n <= 512 ? 512 : 1024;
	PcgKernel const kernel = pick(mixed, s->res_width, precond, nt);
	size_t const lds = static_cast<size_t>(s->res_window) * sizeof(resident::dbl2) + spare(mixed, s->res_width, nt);
	if (lds > 48 * 1024) {
		BFMX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
		                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
	}
	// (tests cut runs into many launches)
	const char* cut = std::getenv("BFMX_RESIDENT_ITERS");
	int64_t const per_launch = cut && std::atoll(cut) > 0 ? std::atoll(cut) : kPerLaunch;
	int64_t const nslots = G > 1 ? 2 * static_cast<int64_t>(G) * kSlotWords : 0;
	int mode = warm ? 1 : 0;
	cap = (cap + kCheckEvery - 1) / kCheckEvery * kCheckEvery;
	while (true) {
		int64_t stop = std::min(cap, (mode == 2 ? out->iter : 0) + per_launch);
		if (G > 1) {
			k_clear<<<static_cast<int>((2 * n + kBlock - 1) / kBlock), kBlock, 0, st>>>(V, 2 * n, nslots);
			Scalars* S = s->d_scal;
			void* args[] = {&V, &mode, &rtol2, &delta2, &stop, &S};
			hipError_t const err = hipLaunchCooperativeKernel(reinterpret_cast<const void*>(kernel), dim3(G), dim3(nt),
			                                                  args, static_cast<unsigned>(lds), st);
			if (err != hipSuccess) {
				(void) hipGetLastError();
				return BFMX_OK;   // the device cannot hold the cluster: the streaming kernels
			}
		} else {
			kernel<<<1, nt, lds, st>>>(V, mode, rtol2, delta2, stop, s->d_scal);
		}
		BFMX_HIP(hipGetLastError());
		BFMX_HIP(hipMemcpyAsync(out, s->d_scal, sizeof(Scalars), hipMemcpyDeviceToHost, st));
		BFMX_HIP(hipStreamSynchronize(st));
		if (out->done == kFailed) {
			return BFMX_OK;
		}
		if (out->done != 0 || out->iter >= cap) {
			*ran = true;
			return BFMX_OK;
		}
		mode = 2;
	}
}

}  // namespace bfmx
