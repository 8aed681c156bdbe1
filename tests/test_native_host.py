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


def test_table_log_accuracy(run_cpp):
    """The expand's FP64 logarithm against 80-bit ones: random values of every exponent, of [0.5, 2], towards
    1 and at the ends of the table's intervals. Half a unit in the last place is the final rounding;
    the series cut after r^9 / 9 (r < 2^-7) leaves 2^-63 / 10 of the result, the rounded parts below
    the high one 2^-59 of it at most: 0.52 in all, and an average of 0.25. Values without a
    normal logarithm go to the library."""
    out = run_cpp(r'''#include <cstdio>
#include <random>
#include "emc_log.h"
int main() {
    std::mt19937_64 g(1);
    auto table_log = [](double x) { return emc::table_log(x, emc::kLogEntries.entry); };
    double worst = 0., sum = 0.;
    long n = 0;
    for (long i = 0; i < 2000000; ++i) {
        const double u = (double)(g() >> 11) * 0x1p-53;
        double x = 0.5 + 1.5 * u;
        if (i % 4 == 1) x = 1. + (u - 0.5) * std::ldexp(1., -(int)(g() % 50));
        if (i % 4 == 2) x = std::ldexp(1. + u, (int)(g() % 2046) - 1022);
        if (i % 4 == 3) {
            const double end = 1. + (double)(g() % 129) / 128.;
            x = __builtin_bit_cast(double, __builtin_bit_cast(long, end) + (long)(g() % 2001) - 1000) * (g() & 1 ? 1. : 0.5);
        }
        const long double want = logl(x);
        if (want == 0.L) {
            if (table_log(x) != 0.) return 1;
            continue;
        }
        int e;
        (void)frexpl(want, &e);
        const double ulp = (double)(fabsl((long double)table_log(x) - want) / ldexpl(1.L, e - 53));
        worst = ulp > worst ? ulp : worst;
        sum += ulp;
        ++n;
    }
    for (double x : {0., -0., 5e-324, 1e-310, 2.2250738585072009e-308, (double)INFINITY, 1.7976931348623157e308})
        if (std::fabs(table_log(x) - std::log(x)) > std::fabs(std::log(x)) * 0x1p-52) return 2;
    for (double x : {-1., -(double)INFINITY, (double)NAN})
        if (table_log(x) == table_log(x)) return 3;
    std::printf("%.6f %.6f\n", worst, sum / (double)n);
}''')
    worst, mean = map(float, out.split())
    assert worst <= 0.52 and mean <= 0.251, out


# What of HIP the engine's buffers call, with a runtime whose last error stays until it is read (as HIP's
# does) and whose allocations fail above a size
FAKE_HIP = r'''#pragma once
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef void *hipStream_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipMemcpyHostToDevice = 1, hipHostMallocDefault = 0 };
inline hipError_t last = hipSuccess;
inline size_t most = 1000;
inline hipError_t hipMalloc(void **p, size_t n) { return n > most ? last = hipErrorOutOfMemory : (*p = malloc(n), hipSuccess); }
inline hipError_t hipHostMalloc(void **p, size_t n, int) { return hipMalloc(p, n); }
inline hipError_t hipFree(void *p) { return free(p), hipSuccess; }
inline hipError_t hipHostFree(void *p) { return hipFree(p); }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
inline hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = *t = most, hipSuccess; }
inline hipError_t hipGetLastError() { const hipError_t e = last; return last = hipSuccess, e; }
inline const char *hipGetErrorString(hipError_t) { return "out of memory"; }
'''


def test_failed_allocation_leaves_no_error(run_cpp, tmp_path):
    """A buffer that gets no memory reports it once and leaves no error for the check after the next launch
    to find: the engine goes on without lists and staging memory that are only there for speed."""
    (tmp_path / 'hip').mkdir()
    (tmp_path / 'hip' / 'hip_runtime_api.h').write_text(FAKE_HIP)
    run_cpp(r'''#include <vector>
#include "emc_host.h"
static int failing_call() {
    HIP_TRY(last = hipErrorOutOfMemory);
    return 0;
}
int main() {
    emc::DevBuf<double> d;
    emc::PinnedBuf<char> h;
    const std::vector<double> v(2000);
    if (d.alloc(10) || hipGetLastError()) return 1;
    if (d.alloc(2000) != EMC_E_NOMEM || d.p || d.n || d.cap) return 2;
    if (emc::g_last_error.find("16000 bytes") == std::string::npos) return 3;
    if (hipGetLastError()) return 4;
    if (d.upload(v.data(), 2000, nullptr) != EMC_E_NOMEM || hipGetLastError()) return 5;
    if (h.reserve(2000) != EMC_E_NOMEM || h.p || hipGetLastError()) return 6;
    if (failing_call() != EMC_E_HIP || hipGetLastError()) return 7;
    if (d.alloc(10) || d.upload(v.data(), 100, nullptr) || h.reserve(10)) return 8;
    // a bad argument asks the runtime nothing
    last = hipErrorOutOfMemory;
    if (emc::fail(EMC_E_ARG, "x") != EMC_E_ARG || hipGetLastError() != hipErrorOutOfMemory) return 9;
    return 0;
}''', '-I%s' % tmp_path)


def test_lists_for_speed_leave_memory_free(run_cpp, tmp_path):
    """alloc_spare takes memory only if `leave` bytes stay free beside it, keeps a large enough buffer, and
    hands a smaller one back before it looks."""
    (tmp_path / 'hip').mkdir()
    (tmp_path / 'hip' / 'hip_runtime_api.h').write_text(FAKE_HIP)
    run_cpp(r'''#include "emc_host.h"
int main() {
    emc::DevBuf<double> d;  // 1000 bytes free
    if (!d.alloc_spare(100, 200) || d.n != 100 || d.cap != 100) return 1;
    if (!d.alloc_spare(50, 100000) || d.n != 50 || d.cap != 100) return 2;
    if (d.alloc_spare(101, 200) || d.p || d.cap) return 3;
    if (d.alloc_spare(1, 1001) || d.alloc_spare((size_t)-1 / 8, 0) || hipGetLastError()) return 4;
    return 0;
}''', '-I%s' % tmp_path)
