"""Which clusters of workgroups run at once (bfm_amd/csrc/hip/cu_budget.h, host
code): what fits the compute units of a shader engine together does, the rest waits in the
order it came, and a launch larger than the device runs alone."""

import os
import subprocess

from bfm_amd import build as B

SOURCE = r"""
#include <atomic>
#include <cassert>
#include <chrono>
#include <thread>
#include <vector>
#include "cu_budget.h"
using bfmx::CuBudget;

static void nap() { std::this_thread::sleep_for(std::chrono::milliseconds(50)); }

int main() {
	assert(CuBudget::share(1) == 1 && CuBudget::share(32) == 1 && CuBudget::share(33) == 2);
	assert(CuBudget::share(224) == 7 && CuBudget::share(225) == 8 && CuBudget::share(256) == 8);
	CuBudget b(256);
	b.take(CuBudget::share(197));
	b.take(CuBudget::share(6));            // fits beside it: returns at once
	std::atomic<int> large{0}, small{0};
	std::thread l([&] { b.take(8); large = 1; b.give(8); });
	nap();
	std::thread s([&] { b.take(1); small = 1; b.give(1); });
	nap();
	assert(!large && !small);              // the large one waits, the later small one behind it
	b.give(1);
	nap();
	assert(!large && !small);
	b.give(7);
	l.join();
	s.join();
	assert(large && small);
	CuBudget tiny(4);                      // fewer compute units than engines: one at a time
	tiny.take(3);
	tiny.give(3);
	// never more than the total
	std::atomic<int> used{0};
	std::vector<std::thread> v;
	for (int k = 0; k < 16; k++) {
		v.emplace_back([&, k] {
			for (int i = 0; i < 200; i++) {
				int const n = 1 + (7 * k + i) % 8;
				b.take(n);
				assert((used += n) <= 8);
				used -= n;
				b.give(n);
			}
		});
	}
	for (auto& t : v) t.join();
}
"""


def test_budget(tmp_path):
    src, exe = tmp_path / "t.cc", tmp_path / "t"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(B.HIP_DIR), str(src), "-o", str(exe)],
                   check=True)
    subprocess.run([str(exe)], check=True, timeout=60)
