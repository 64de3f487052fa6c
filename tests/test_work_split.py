"""The split of a work queue over waves (csrc/mtx_split.h), compiled for the
host: every entry belongs to one chunk, up to the largest 32-bit count."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "mtx_split.h"
int main(int argc, char **argv) {
  for (int i = 1; i + 1 < argc; i += 2) {
    const uint32_t n = strtoul(argv[i], nullptr, 10), w = strtoul(argv[i + 1], nullptr, 10);
    const uint32_t c = mtx::queue_chunk(n, w);
    std::printf("%u %u %u\\n", mtx::queue_lanes(n, w), c, mtx::queue_chunks(n, c));
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("split")
    (d / "split.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mutracer_amd", "csrc"),
                    str(d / "split.cpp"), "-o", str(d / "split")], check=True)
    return str(d / "split")


@pytest.mark.parametrize("waves", [16, 5120, 7168])
def test_every_entry_in_one_chunk(program, waves):
    top = 2**32
    counts = [1, 2, 63, 64, 65, waves - 1, waves, waves + 1, 64 * waves, 64 * waves + 1, 512 * waves * 2,
              512 * waves * 9 + 1, top - 257, top - 256, top - 255, top - 64, top - 63, top - 1]
    args = [str(x) for n in counts for x in (n, waves)]
    out = subprocess.run([program] + args, check=True, capture_output=True, text=True).stdout.split("\n")
    for n, line in zip(counts, out):
        lanes, chunk, chunks = map(int, line.split())
        assert lanes == min(64, max(1, -(-n // waves)))
        assert chunk >= lanes and chunk <= 256
        assert (chunks - 1) * chunk < n <= chunks * chunk, (n, chunk, chunks)


def test_wave_barriers_order_memory():
    """The bare wave barrier orders no memory: lanes that hand values to one
    another through LDS meet in wave_sync(), its only user."""
    csrc, uses = os.path.join(ROOT, "mutracer_amd", "csrc"), []
    for f in sorted(os.listdir(csrc)):
        if f.endswith((".h", ".hip", ".cpp")):
            text = open(os.path.join(csrc, f)).read()
            uses += [f] * text.count("__builtin_amdgcn_wave_barrier(")
    assert uses == ["mtx_fetch.h"]
