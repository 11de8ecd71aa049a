"""The store of a search state after a transition (gctf_internal.hpp,
step_store), run on the CPU: the lanes of the wavefront that calls it have no
order among themselves, so every order has to leave the same state -- the new
values where the transition holds them, the previous state's elsewhere."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gctffind_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <hip/hip_runtime.h>
#include "gctf_internal.hpp"
using namespace gctf;

constexpr int W = sizeof(SearchState) / 4;
static void fill(SearchState& s, int base)
{
	int w[W];
	for (int i = 0; i < W; ++i) w[i] = base + i;
	memcpy(&s, w, sizeof s);
}

int main()
{
	SearchState in, fresh, held, got;
	fill(in, 1000);
	fill(fresh, 2000);
	int want[W], back[W], bad = 0, held_words = 0;
	// the words that a transition holds: those that step_fields carries over
	fill(held, 3000);
	step_fields(held, fresh);
	int hw[W], fw[W], iw[W];
	memcpy(hw, &held, sizeof held); memcpy(fw, &fresh, sizeof fresh); memcpy(iw, &in, sizeof in);
	for (int i = 0; i < W; ++i) {
		const bool h = hw[i] == fw[i];
		held_words += h;
		want[i] = h ? fw[i] : iw[i];
	}
	for (int order = 0; order < 64; ++order) {
		fill(got, 4000);
		// lane `order` first, then the others upwards, or all downwards
		if (order == 63) {
			for (int l = 63; l >= 0; --l) step_store(&got, &in, fresh, l);
		} else {
			for (int k = 0; k < 64; ++k) step_store(&got, &in, fresh, (order + k) & 63);
		}
		memcpy(back, &got, sizeof got);
		for (int i = 0; i < W; ++i)
			if (back[i] != want[i]) {
				printf("order %d word %d: %d, not %d\n", order, i, back[i], want[i]);
				++bad;
			}
		// in place
		SearchState self = in;
		for (int k = 0; k < 64; ++k) step_store(&self, &self, fresh, (order + k) & 63);
		memcpy(back, &self, sizeof self);
		for (int i = 0; i < W; ++i) bad += back[i] != want[i];
	}
	printf("%d of %d words held, %d wrong\n", held_words, W, bad);
	return bad != 0;
}
"""


def test_state_store_in_any_lane_order(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src, exe = tmp_path / "state.hip", tmp_path / "state"
    src.write_text(PROGRAM)
    cmd = [hipcc, "--offload-host-only", "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[:2000]
