"""Host parts of the engine's sources that need no GPU, compiled with g++ and run here."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'dragonfly_amd', 'csrc')


@pytest.fixture
def run_cpp(tmp_path):
    """Compile a C++ program against the engine's headers and return what it prints."""
    def run(source, *flags):
        src, exe = tmp_path / 'prog.cpp', tmp_path / 'prog'
        src.write_text(source)
        subprocess.run(['g++', '-std=c++17', '-O2', '-ffp-contract=off', '-I' + CSRC, str(src), '-o', str(exe),
                        *flags], check=True)
        return subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return run


# (tiles, blocks a tile): one launch; 3208 tiles of 4180 quarter patches (13.4 million blocks, one launch)
# and 257,000, 512,000 and 2 million slots of the same detector (past 2^24 blocks of 256 work-items);
# tiles that alone fill a launch
@pytest.mark.parametrize('tiles, per_tile', ((1, 1), (7, 28), (3208, 4180), (4016, 4180), (8000, 4180), (8003, 4180),
                                             (32000, 4180), (24, 2000000), (0, 5)))
def test_tile_spans_fit_a_grid(run_cpp, tiles, per_tile):
    """The spans cover every tile once, in order, start at whole groups of XCDs, and no launch reaches the
    2^32 work-items at which a grid wraps."""
    out = run_cpp('''#include <cstdio>
#include "emc_grid.h"
int main() {
    emc::for_each_tile_span(%d, 8, %d, 256, [](long first, long count, unsigned blocks) {
        std::printf("%%ld %%ld %%u\\n", first, count, blocks);
    });
}''' % (tiles, per_tile))
    spans = [tuple(map(int, line.split())) for line in out.splitlines()]
    at = 0
    for first, count, blocks in spans:
        assert first == at and first % 8 == 0 and count > 0
        assert blocks == -(-count // 8) * 8 * per_tile and blocks * 256 < 1 << 32
        at += count
    assert at == tiles
    if -(-tiles // 8) * 8 * per_tile < 1 << 24:
        assert len(spans) == (tiles > 0)
