"""The plan of a split dK/dV grid (csrc/gfa_plan.h), compiled for the host with g++: the chunk it picks
is the one a plain list schedule of every candidate's workgroups picks, its workgroup count is the
sum of the split counts that the kernels derive from the chunk (a difference would leave rows of
dK and dV unwritten), and planning allocates no memory (it runs inside C entry points)."""
import heapq
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gemma-triton-flash-attn_amd", "csrc")

PROG = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include "gfa_plan.h"
static long allocations = 0;
void* operator new(size_t n) { ++allocations; return malloc(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
int main() {
  int B, Hkv, R, N, causal, window, wkv, wgs, qs;
  while (scanf("%d %d %d %d %d %d %d %d %d", &B, &Hkv, &R, &N, &causal, &window, &wkv, &wgs, &qs) == 9) {
    gfa::BwdDkvParams p{};
    p.B = B; p.Hkv = Hkv; p.Hq = R * Hkv; p.R = R; p.N = N; p.causal = causal; p.window = window;
    p.wkv = wkv; p.n_kb = (N + wkv - 1) / wkv; p.q_splits = qs;
    const long before = allocations;
    const gfa::DkvPlan plan = gfa::plan_dkv(p, wgs);
    const long made = allocations - before;
    p.chunk = plan.chunk;
    long long sum = 0;
    for (int kb = 0; kb < p.n_kb; ++kb) sum += gfa::dkv_splits(p, kb * wkv);
    printf("%d %d %lld %ld\n", plan.chunk, plan.nblocks, sum * B * Hkv, made);
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def plan_prog(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("dkvplan")
    src = d / "dkv_plan.cpp"
    src.write_text(PROG)
    exe = d / "dkv_plan"
    subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-D__host__=", "-D__device__=", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return str(exe)


def _iterations(R, N, causal, window, wkv):
    """Query tiles x heads that see each key block (the dK/dV kernel's loop)."""
    nq, out = (N + 31) // 32, []
    for k0 in range(0, N, wkv):
        last = min(N, k0 + wkv) - 1
        hi = min(nq, (last + window - 1) // 32 + 1) if causal and window else nq
        out.append(R * (hi - (k0 // 32 if causal else 0)))
    return out


def _plan(B, Hkv, R, N, causal, window, wkv, wgs, qs):
    its, copies, slots = _iterations(R, N, causal, window, wkv), B * Hkv, 256 * wgs

    def splits(chunk):
        return [qs if chunk == 0 else max(1, min(qs, -(-n // chunk))) for n in its]

    def cost(chunk):
        free, end, partials = [0] * slots, 0, 0
        for n, c in zip(its, splits(chunk)):
            partials += c * copies if c > 1 else 0
            for _ in range(c * copies):
                t = heapq.heappop(free) + -(-n // c) + 8
                end = max(end, t)
                heapq.heappush(free, t)
        return end + 0.03 * partials

    best, best_cost = 0, cost(0)
    longest = max(1, max(its))
    for halves in (2, 3, 4):
        lo, hi = -(-longest // qs), longest
        while lo < hi:
            mid = (lo + hi) // 2
            if sum(splits(mid)) * copies <= slots * halves // 2:
                hi = mid
            else:
                lo = mid + 1
        c = cost(lo)
        if c < best_cost:
            best, best_cost = lo, c
    return best


SHAPES = [(B, Hkv, R, N, causal, window, wkv, wgs, qs)
          for N in (1, 33, 97, 333, 800, 1709, 2001, 3000, 5000, 16384)
          for causal, window in ((1, 0), (0, 0), (1, 37), (1, 512), (1, 1024)) if window < N
          for B, Hkv, R in ((1, 1, 8), (1, 4, 2), (2, 2, 8), (3, 2, 3), (1, 16, 1))
          for wkv, wgs in ((64, 1), (128, 1), (64, 2), (128, 2))
          for qs in (2, 4, 8) if -(-N // wkv) * B * Hkv * qs <= 2048]


def _run(prog, shapes):
    text = "\n".join(" ".join(map(str, s)) for s in shapes)
    out = subprocess.run([prog], input=text, check=True, capture_output=True, text=True).stdout.split("\n")
    return [tuple(map(int, line.split())) for line in out if line]


def test_same_as_list_schedule(plan_prog):
    got = _run(plan_prog, SHAPES)
    assert len(got) == len(SHAPES)
    for shape, (chunk, blocks, total, allocations) in zip(SHAPES, got):
        assert chunk == _plan(*shape), shape
        assert allocations == 0 and (chunk == 0 or blocks == total), (shape, blocks, total, allocations)


def test_large_grids(plan_prog):
    """More key blocks than the plan holds keep equal splits; workgroups longer than its time axis are
    planned in coarser steps (non-causal work is uniform: one split each where the grid is full)."""
    big = [(1, 1, 8, 140000, 1, 0, 128, 2, 2), (1, 1, 1, 1 << 20, 1, 0, 64, 1, 8), (1, 1, 64, 32556, 0, 0, 128, 1, 2),
           (1, 1, 64, 131072, 1, 0, 128, 2, 2), (33000, 1, 1, 64, 1, 0, 128, 2, 8)]
    got = _run(plan_prog, big)
    assert [g[0] for g in got[:3]] == [0, 0, 64 * ((32556 + 31) // 32)]
    assert all(a == 0 and (c == 0 or b == t) for c, b, t, a in got)
