"""A prepared differentiable context goes on without what it only keeps for speed when memory runs out: the
choice (vulkanexp_amd/csrc/diff_memory.hpp) compiled against an allocator with a limit."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r'''
#include <cstdio>
#include <cstdlib>
#include "diff_memory.hpp"
int main(int, char** argv) {
	size_t left = std::strtoull(argv[3], nullptr, 10), at = 0;
	const ddgi::DiffSpare m = ddgi::diff_spare_memory(std::strtoull(argv[1], nullptr, 10), std::strtoull(argv[2], nullptr, 10),
		[&](size_t bytes) -> void* {
			if(bytes > left) return nullptr;
			left -= bytes;
			return reinterpret_cast<void*>(++at);
		});
	std::printf("%d %u %d\n", m.keys != nullptr, m.taps, m.records != nullptr);
}
'''


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("diff_memory")
    (d / "p.cpp").write_text(PROGRAM)
    cmd = ["g++", "-std=c++17", "-Wall", "-o", str(d / "p"), str(d / "p.cpp"),
           "-I" + os.path.join(ROOT, "vulkanexp_amd", "csrc")]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return str(d / "p")


N, P = 100_000, 1000
TAPS, ONE, RECORDS = 768 * P, 12 * P, 80 * N


@pytest.mark.parametrize("texels,probes,memory,want", [
    (N, P, TAPS + RECORDS, "1 64 1"),
    (N, P, TAPS + RECORDS - 1, "1 64 0"),            # the records do not fit
    (N, P, TAPS - 1, "1 1 0"),                       # nor do the counters per tap
    (N, P, ONE, "1 1 0"),
    (N, P, ONE - 1, "0 1 0"),                        # refused
    ((12 << 20) + 1, P, 1 << 40, "1 64 0"),          # too many texels for records
    (N, (1 << 18) + 1, 1 << 40, "1 1 1"),            # too many probes for counters per tap
])
def test_what_is_left_out(program, texels, probes, memory, want):
    r = subprocess.run([program, str(texels), str(probes), str(memory)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == want
