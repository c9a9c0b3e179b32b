"""k_l1_scan on the CPU: its own source text (bucket.hip), one fiber per thread, the threads
between two barriers run one after the other in ascending or descending order.  Offsets, block
table and status are fixed by the counts, so every order has to give them, whatever the
workspace held before the call."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lofar_amd",
                    "csrc")

HOST = r"""
#include <ucontext.h>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include <algorithm>
#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(x)
#define __shared__ static
#define __threadfence_system()
using std::min;
struct Dim { int x; };
static Dim threadIdx;
struct int2 { int x, y; };
constexpr int NT = 1024;
static ucontext_t sched, fib[NT];
static long long lanes[NT];
static void __syncthreads()
{
    const int t = threadIdx.x;
    swapcontext(&fib[t], &sched);
    threadIdx.x = t;
}
template <typename T>
static T __shfl_up(T v, int d, int)
{
    const int t = threadIdx.x;
    lanes[t] = v;
    __syncthreads();
    const T r = (T)lanes[(t & 63) >= d ? t - d : t];
    __syncthreads();
    return r;
}
template <typename T>
static T atomicAdd(T* p, T v) { const T o = *p; *p += v; return o; }
static unsigned atomicMax(unsigned* p, unsigned v) { const unsigned o = *p; *p = std::max(o, v); return o; }
"""

MAIN = r"""
static long long nk1, bs, n_blk;
static unsigned *c1, *ce;
static long long *off1, *eoff1, *boff;
static L2Block* blk;
static long long status[4];
static int err = 5, done;
static void thread()
{
    k_l1_scan(nk1, c1, ce, off1, eoff1, bs, boff, blk, &err, status, 77, Heavy());
    done++;
    swapcontext(&fib[threadIdx.x], &sched);
}
int main(int argc, char** argv)
{
    const bool down = atoi(argv[1]);
    const long long stale = atoll(argv[2]);
    bs = atoll(argv[3]);
    if (scanf("%lld %lld", &nk1, &n_blk) != 2) return 1;
    std::vector<unsigned> a(nk1), b(nk1);
    for (auto& x : a) if (scanf("%u", &x) != 1) return 1;
    for (auto& x : b) if (scanf("%u", &x) != 1) return 1;
    std::vector<long long> o(nk1 + 1, stale), e(nk1 + 1, stale), f(nk1 + 1, stale);
    std::vector<L2Block> k(n_blk + 1, L2Block{-1, -1, -1, -1});
    c1 = a.data(); ce = b.data(); off1 = o.data(); eoff1 = e.data(); boff = f.data(); blk = k.data();
    std::vector<std::vector<char>> stack(NT, std::vector<char>(64 << 10));
    for (int t = 0; t < NT; t++) {
        getcontext(&fib[t]);
        fib[t].uc_stack.ss_sp = stack[t].data();
        fib[t].uc_stack.ss_size = stack[t].size();
        fib[t].uc_link = &sched;
        makecontext(&fib[t], thread, 0);
    }
    while (done < NT)  // one turn of every thread up to its next barrier
        for (int i = 0; i < NT; i++) {
            threadIdx.x = down ? NT - 1 - i : i;
            swapcontext(&sched, &fib[threadIdx.x]);
        }
    for (long long v : o) printf("%lld ", v);
    puts("");
    for (long long v : e) printf("%lld ", v);
    puts("");
    for (auto& d : k) printf("%lld %lld %lld ", d.k1, d.beg, d.end);
    puts("");
    for (long long v : status) printf("%lld ", v);
    puts("");
}
"""


def block(text, head):
    """The source from `head` (a regular expression) to the closing brace of its body."""
    m = re.search(head, text)
    assert m, head
    at = text.index("{", m.start())
    depth = 0
    for i in range(at, len(text)):
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        if depth == 0:
            return text[m.start():i + 1] + (";" if text[i + 1] == ";" else "") + "\n"
    raise AssertionError(head)


@pytest.fixture(scope="module")
def scan(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    hdr = open(os.path.join(CSRC, "grid_kernels.h")).read()
    src = open(os.path.join(CSRC, "bucket.hip")).read()
    code = HOST
    for s in ("L2Block", "HeavyTile", "HeavyState", "Heavy"):
        code += block(hdr, r"struct (alignas\(32\) )?%s \{" % s)
    for f in ("T block_exscan", "void list_heavy", "void clear_heavy"):
        code += block(src, r"(template <[^>]*>\n)?__device__ __forceinline__ " + f)
    code += block(src, r"__global__ __launch_bounds__\(1024\) void k_l1_scan") + MAIN
    d = tmp_path_factory.mktemp("scan")
    (d / "scan.cpp").write_text(code)
    subprocess.run([cxx, "-O1", "-std=c++17", "-w", "-o", str(d / "scan"), str(d / "scan.cpp")],
                   check=True)
    return str(d / "scan")


@pytest.mark.parametrize("down", [0, 1])
@pytest.mark.parametrize("stale", [0, 1 << 40])
@pytest.mark.parametrize("nk1,last", [(1, 5000), (7, 1), (1024, 3000), (1025, 2048), (2500, 0)])
def test_offsets_blocks_and_status(scan, nk1, last, down, stale):
    bs = 1024
    rng = np.random.default_rng(nk1)
    rec = rng.integers(0, 3000, nk1) * (rng.random(nk1) < 0.5)
    rec[-1] = last
    ent = rec * 2
    off = np.concatenate([[0], np.cumsum(rec)])
    want = [(k, b, min(off[k + 1], b + bs)) for k in range(nk1)
            for b in range(off[k], off[k + 1], bs)]
    feed = "%d %d\n%s\n%s\n" % (nk1, len(want), " ".join(map(str, rec)), " ".join(map(str, ent)))
    out = subprocess.run([scan, str(down), str(stale), str(bs)], input=feed, text=True,
                         capture_output=True, check=True, timeout=60).stdout.splitlines()
    o, e, k, st = [np.array(x.split(), dtype=np.int64) for x in out]
    assert np.array_equal(o, off) and np.array_equal(e, 2 * off)
    assert np.array_equal(k.reshape(-1, 3)[:-1], np.array(want).reshape(-1, 3))
    assert (k.reshape(-1, 3)[-1] == -1).all()  # nothing past the table
    assert st[0] == 2 * off[-1] and st[1] == 5 and st[2] == 77
