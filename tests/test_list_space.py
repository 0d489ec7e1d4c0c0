"""Arithmetic of the block lists' space (lucid_amd/csrc/list_space.h), compiled for the host: frames
near and beyond the 2^32 entries that a block slot can address, which no test could fill."""

import os
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lucid_amd", "csrc",
                      "list_space.h")

PROGRAM = r"""
#include "list_space.h"
#include <assert.h>
#include <stdio.h>
using namespace lucid;

int main() {
	const uint64_t low = 2040ull * 16 * 256;
	// fixed high bins of `fixed` positions, then `n` promoted ones of 1000 each
	const uint32_t sizes[] = {0u, 1000u, 262144u, (1u << 28) - 600000u, 1u << 28, 0xffffffffu};
	const uint64_t caps[] = {low, low + (1ull << 22), 1ull << 32};
	for(uint32_t fixed : sizes)
		for(uint64_t cap : caps) {
			const bool fixed_fit = lists_fit(low, 0u, fixed, cap);
			assert(fixed_fit == (low + 16ull * fixed <= cap));
			uint32_t cursor = list_cursor_start(fixed);
			uint64_t end = low + 16ull * fixed; // of the lists so far
			bool all = fixed_fit;
			for(int n = 0; n < 5120; n++) {
				const uint32_t at = cursor;
				cursor += 1000u;
				assert(cursor > at); // the cursor does not wrap
				const bool ok = lists_fit(low, at, 1000u, cap);
				all = all && ok;
				if(fixed_fit) {
					// a promoted bin's lists follow all others', in the slots' 32 bits where they fit
					assert(list_entry(low, at) == end);
					assert(ok == (end + 16000ull <= cap));
					assert(!ok || (uint32_t)list_entry(low, at) == end);
					end += 16000ull;
				} else {
					assert(!ok); // nor does anything behind lists that do not fit
				}
			}
			if(all)
				continue;
			// the lists grow once to what the frame needs, or cannot
			const uint64_t need = low + 16ull * cursor, grown = grown_list_cap(low, cursor, cap);
			assert(need > kMaxListEntries ? grown == 0 : grown >= need && grown <= kMaxListEntries);
			if(need <= kMaxListEntries)
				assert(grown > cap || cap == kMaxListEntries);
		}
	puts("ok");
}
"""


@pytest.fixture(scope="module")
def compile_and_run(tmp_path_factory):
    def run(source):
        d = tmp_path_factory.mktemp("list_space")
        (d / "main.cpp").write_text(source)
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.dirname(HEADER), "-o",
                        str(d / "main"), str(d / "main.cpp")], check=True)
        return subprocess.run([str(d / "main")], capture_output=True, text=True)
    return run


def test_cursor_and_offsets(compile_and_run):
    out = compile_and_run(PROGRAM)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stderr


GROWING = r"""
#include "list_space.h"
#include <stdio.h>
using namespace lucid;

int main() {
	// a scene whose lists grow by 5 % a frame, to about 300 times the first space
	const uint64_t low = 2040ull * 16 * 256;
	uint64_t cap = low + (1ull << 22);
	int frames = 0, overflows = 0;
	for(double p = 200000.0; p < 60e6; p *= 1.05, frames++)
		if(!lists_fit(low, 0u, (uint32_t)p, cap)) {
			overflows++;
			cap = grown_list_cap(low, (uint32_t)p, cap);
			if(!lists_fit(low, 0u, (uint32_t)p, cap))
				return 1;
		}
	printf("%d %d\n", frames, overflows);
}
"""


def test_a_growing_scene_overflows_seldom(compile_and_run):
    """Doubling: at most one overflow for every factor of two, log2(300) of them."""
    out = compile_and_run(GROWING)
    frames, overflows = map(int, out.stdout.split())
    assert out.returncode == 0 and frames > 100 and 0 < overflows <= 9
