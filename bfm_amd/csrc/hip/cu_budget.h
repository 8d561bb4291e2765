// Which clusters of workgroups run at once on a device.
//
// The workgroups of a cluster wait for each other, so all of them must become
// resident, whatever else runs. The hardware deals a launch's workgroups in turn
// to the 32 shader engines (the eight XCDs first, the four engines of each then),
// beginning with the same one, and one that is full keeps its workgroup waiting
// although another has room: beside a launch of 224 workgroups of 1,024 threads
// (seven of an engine's eight compute units) another of 6, 8 or 16 starts at
// once, beside one of 225 only when that ends. So a launch of G takes ceil(G / 32)
// compute units of an engine at most, and while the sum of that over the launches
// at hand is no more than an engine has, there is a compute unit for every
// workgroup (it needs one at most; kernels that do not wait end and leave theirs).
// Clusters of several threads then run beside each other. A launch that does not
// fit waits; they are served in the order they came, so that small ones do not keep
// a large one waiting forever.
// Measured: a 5,124-node solve (six workgroups) beside solves of 201,051 nodes
// (197), with one launch at a time 39.5 ms, here 4.2 ms; eight threads of 5,124
// nodes 4.2 ms a solve, here 1.6.
#pragma once

#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace bfmx {

class CuBudget {
public:
	static constexpr int kEngines = 32;

	explicit CuBudget(int compute_units) : m_total(compute_units / kEngines) {}

	// Compute units of an engine that a launch of G workgroups takes at most.
	static int share(int64_t G) {
		return static_cast<int>((G + kEngines - 1) / kEngines);
	}

	// Waits until n fit beside what is taken (a launch alone always does).
	void take(int n) {
		std::unique_lock<std::mutex> lock(m_mutex);
		uint64_t const turn = m_next++;
		m_changed.wait(lock, [&] { return m_turn == turn && (m_used == 0 || m_used + n <= m_total); });
		m_used += n;
		m_turn++;
		m_changed.notify_all();
	}

	void give(int n) {
		std::lock_guard<std::mutex> const lock(m_mutex);
		m_used -= n;
		m_changed.notify_all();
	}

private:
	std::mutex m_mutex;
	std::condition_variable m_changed;
	int const m_total;
	int m_used = 0;
	uint64_t m_next = 0, m_turn = 0;
};

}  // namespace bfmx
