"""CPU unit tests of host-library pieces that need no GPU.

The copy-pool partition (csrc/fa_copy_parts.h) decides which bytes of a
host-slice upload or download each host thread copies.  A partition that
leaves a gap sends stale bytes of the pinned ring to the device, so every
byte count -- in particular the odd 16-bit ones, 2 * (128m + 1) -- must be
covered exactly once.  The header is compiled here with g++ on its own.

The launch planner's fold and few_rows flags, which pick a body or a row order
inside a kernel and so do not show in its name or grid, are read from
csrc/fa_host.cpp itself for the shapes of the GPU tests that mean to run them.

Also the arithmetic behind one 16-bit GPU test input (f16 probabilities in
the subnormal range).
"""
from __future__ import annotations

import os
import subprocess

import numpy as np

import test_gpu_fold
import test_gpu_lp_rows
import test_gpu_lp_wide
from fa_testutil import long_row_f16_case

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "flash-attention-cpu_amd", "csrc")

CHECK = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "fa_copy_parts.h"

// Every byte of [0, n) covered by exactly one part, parts in order, each
// part starting on a 64-byte boundary.
static int check(size_t n, int parts) {
    size_t next = 0;
    for (int id = 0; id < parts; ++id) {
        size_t b, len;
        fa_copy_part_range(n, parts, id, &b, &len);
        if (len == 0) continue;
        if (b != next || b % 64 != 0 || b + len > n) {
            std::printf("bad part n=%zu parts=%d id=%d b=%zu len=%zu next=%zu\n", n, parts, id, b, len, next);
            return 1;
        }
        next = b + len;
    }
    if (next != n) {
        std::printf("gap n=%zu parts=%d covered=%zu\n", n, parts, next);
        return 1;
    }
    return 0;
}

int main() {
    int bad = 0;
    std::vector<size_t> ns = {0, 1, 2, 63, 64, 65, 255, 256, 257, 1053954, 8388614, (size_t)16 << 20};
    // n = 256m + r for r = 1, 2, 3 (odd 16-bit element counts give r = 2),
    // small m and m around the 1 MiB threading cut and the 16 MiB chunk.
    for (size_t m : {1ul, 2ul, 3ul, 100ul, 4095ul, 4096ul, 4117ul, 4118ul, 65535ul, 65536ul})
        for (size_t r : {1ul, 2ul, 3ul}) ns.push_back(256 * m + r);
    for (size_t n = 0; n < 4096; ++n) ns.push_back(n);
    for (size_t n : ns)
        for (int parts = 1; parts <= 8; ++parts) bad |= check(n, parts);
    std::printf(bad ? "FAIL\n" : "OK\n");
    return bad;
}
"""


def test_copy_pool_partition_covers_every_byte(tmp_path):
    src = tmp_path / "check_parts.cpp"
    exe = tmp_path / "check_parts"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout


PLAN = r"""
#include "fa_host.cpp"
int fa_scratch_init(int) { return FA_ERR_SCRATCH; }
void* fa_scratch_ptr(int) { return nullptr; }

// stdin: variant dtype bh sq sk d causal; stdout: fold few_rows kernel
int main() {
    int variant, dtype, causal;
    size_t bh, sq, sk, d;
    static const float dummy[4] __attribute__((aligned(16))) = {0, 0, 0, 0};
    while (std::scanf("%d %d %zu %zu %zu %zu %d", &variant, &dtype, &bh, &sq, &sk, &d, &causal) == 7) {
        fa_launch_opts opts = {0.0f, FA_PATH_AUTO, 0, dtype};
        Plan plan;
        if (make_plan(variant, dummy, dummy, dummy, dummy, bh, sq, sk, d, causal, &opts, 256, &plan) != FA_OK) return 1;
        std::printf("%d %d %s\n", plan.p.fold, plan.p.few_rows, plan.first.name.c_str());
    }
    return 0;
}
"""


def test_plans_fold_and_stream_rows_where_the_gpu_tests_say(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PLAN)
    subprocess.run([os.path.join(rocm, "llvm", "bin", "clang++"), "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(rocm, "include"), "-I", CSRC, str(src), "-L", os.path.join(rocm, "lib"),
                    "-lamdhip64", "-Wl,-rpath," + os.path.join(rocm, "lib"), "-lpthread", "-ldl", "-o", str(exe)],
                   check=True)
    calls = [((v, 0, *s, 1), (1, 0)) for s in test_gpu_fold.FOLD for v in (2, 3)]
    calls += [((2, dt, *s, 0), (0, 1)) for s in test_gpu_lp_rows.SHAPES for dt in (1, 2)]
    calls += [((2, dt, *s[1:5], int(s[5])), (int(s[5]), 0)) for s in test_gpu_lp_wide.SHAPES for dt in (1, 2)]
    # neither: the key split by the streaming body's kernel name, more rows, few keys, unfolded small blocks
    calls += [((2, 1, 6, 32, 1416, 128, 0), (0, 0)), ((2, 1, 8, 48, 4096, 128, 0), (0, 0)),
              ((2, 1, 8, 16, 255, 128, 0), (0, 0)), ((3, 0, 32, 2048, 2048, 120, 1), (0, 0)),
              ((1, 0, 128, 256, 256, 64, 1), (0, 0)), ((2, 1, 114, 210, 210, 128, 1), (0, 0))]
    text = "".join(" ".join(str(x) for x in c) + "\n" for c, _ in calls)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(out) == len(calls)
    for (call, flags), line in zip(calls, out):
        assert tuple(int(x) for x in line.split()[:2]) == flags, (call, line)


def test_long_row_f16_case_breaks_the_bound_without_scaling():
    """CPU check of fa_testutil.long_row_f16_case (run on the GPU by
    test_gpu_lp.py): the small probability as the 16-bit kernel forms it
    (exp2((s - m) c) in f32), rounded to f16 directly, misses the 16-bit
    bound; rounded as 2^7 p, as the kernel now does, it stays inside."""
    q, k, v, sq, sk, d = long_row_f16_case()
    c = np.float32(np.float32(1.0 / np.sqrt(np.float32(d))) * np.float32(1.4426950408889634))
    s1 = np.float32(4.0) * np.float32(k[d])   # q . k_j for j >= 1
    t = np.exp2((s1 - np.float32(48.0)) * c, dtype=np.float32)
    assert np.float32(2.0 ** -24) < t < np.float32(2.0 ** -14)   # subnormal in f16
    n = sk - 1

    def out(p):   # O column with every p_j = p (key 0: p = 1), V = -1 / +1
        return (-1.0 + n * p) / (1.0 + n * p)

    exact = out(float(t))
    u = 2.0 ** -11
    bound = u / (1.0 - u) + 2e-5   # the 16-bit bar at max|V| = 1
    direct = out(float(np.float16(t)))
    scaled = out(float(np.float16(t * np.float32(128.0))) / 128.0)
    assert abs(direct - exact) > 2.5 * bound
    assert abs(scaled - exact) < 0.5 * bound
