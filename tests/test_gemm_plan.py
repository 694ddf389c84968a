"""The GEMM kernels' host-checkable rules on the CPU.  The operand-tile plan:
what the kernel addresses lies inside the workspace that the plan sizes (a
small host program includes the kernel's own addressing, gemm_tiled.h, and
asks the built library for plans).  The copies into LDS that are issued as
inline assembly: a wait state between the write of M0 and the load."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "yule_amd" / "csrc"

SCALE_WALK = r"""
#include <cstdio>
#include "gemm_tiled.h"
using namespace yule;
// the last scale row that any walk over stages [s_lo, total) copies, for every start
int main() {
    const uint32_t dts[] = {YULE_DTYPE_Q4_K, YULE_DTYPE_Q5_K, YULE_DTYPE_Q6_K, YULE_DTYPE_Q8_K, YULE_DTYPE_Q8_0, YULE_DTYPE_Q4_0};
    const uint32_t shapes[][3] = {{1, 1, 256}, {3, 31, 512}, {129, 257, 1024}, {2, 134000, 512}, {700, 14336, 4096},
                                  {1000, 4096, 14336}, {130, 67000, 1024}};
    for (uint32_t dt : dts)
        for (auto &sh : shapes)
            for (int f32 = 0; f32 < 2; f32++) {
                TiledPlan p;
                if (!gemm_tiled_plan(sh[0], sh[1], sh[2], dt, f32, &p)) continue;
                const uint32_t k = sh[2], main_s = k / 32, total = main_s + p.ext / 32, np = (p.n_chunk + 255) / 256 * 256;
                for (uint32_t s_lo = 0; s_lo < total; s_lo += 8) {
                    uint32_t row = tile_scale_row(p.gran, s_lo, main_s), fs = s_lo, last = 0;
                    for (;;) {
                        const uint32_t want = tile_scale_row(p.gran, fs, main_s);
                        if (row != want) { printf("type %u k %u stage %u: row %u, not %u\n", dt, k, fs, row, want); return 1; }
                        if (row + tile_scale_rows(p.gran) > last) last = row + tile_scale_rows(p.gran);
                        if (fs + 1 >= total) break;
                        fs++;
                        row += tile_scale_step(p.gran, fs, main_s);
                    }
                    if ((size_t)last * np * 4 > p.s_bytes) { printf("type %u k %u: row %u past the scales\n", dt, k, last); return 1; }
                }
                printf(".");
            }
    printf("\n");
    return 0;
}
"""

# the tests' wide products: bytes of tail partials and passes, on the 256 CUs of the target
TAILS = r"""
#include <cstdio>
#include "gemm_tiled.h"
using namespace yule;
int main() {
    const uint32_t c[][5] = {CASES};
    for (auto &x : c) {
        TiledPlan p;
        if (!gemm_tiled_plan(x[1], x[2], x[3], x[0], x[4], &p)) { printf("none "); continue; }
        printf("%zu:%u ", p.t_bytes, (x[2] + p.n_chunk - 1) / p.n_chunk);
    }
    printf("\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def host_run(tmp_path_factory):
    if shutil.which("g++") is None or not Path("/opt/rocm/include/hip/hip_runtime.h").exists():
        pytest.skip("no host compiler or HIP headers")
    d = tmp_path_factory.mktemp("plan")

    def go(name, source, **env):
        src, exe = d / f"{name}.cpp", d / name
        src.write_text(source)
        subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", "-I/opt/rocm/include", str(src),
                        "-o", str(exe), str(ROOT / "yule_amd" / "libyule_hip.so"), f"-Wl,-rpath,{ROOT / 'yule_amd'}",
                        "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"], check=True)
        return subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, env={"PATH": "/usr/bin:/bin", **env})

    return go


def test_scale_rows_stay_inside_the_scales(host_run):
    r = host_run("scales", SCALE_WALK, YULE_GEMM_TILED_MIN="1")
    assert r.returncode == 0 and r.stdout.count(".") >= 35, r.stdout + r.stderr


def test_wide_cases_have_tail_tiles(host_run):
    """The shapes that stand for the tail tiles (gemm_tiled_check.py's of 1024
    and 1536 columns, test_runner_prefill_tail_tiles's output product) have
    some, in one pass and in two."""
    from gemm_tiled_check import WIDE
    from yule_amd import DType
    cases = [(int(dt), m, n, k, 1) for dt, m, n, k in WIDE if k in (1024, 1536)] + [(int(DType.Q4_K), 2100, 8192, 8192, 1)]
    r = host_run("tails", TAILS.replace("CASES", ", ".join("{%d, %d, %d, %d, %d}" % c for c in cases)), YULE_GEMM_TILED_MIN="1")
    got = [tuple(int(v) for v in w.split(":")) for w in r.stdout.split()]
    assert len(got) == len(cases) == 4 and all(t > 0 for t, _ in got), r.stdout + r.stderr
    assert [n for _, n in got] == [1, 1, 2, 1]


def test_wait_state_between_m0_and_lds_loads():
    """gfx9: one wait state between a scalar write of M0 and a load into LDS;
    the compiler adds it for its own loads and does not look into asm text."""
    found = 0
    for src in sorted([*CSRC.glob("*.hip"), *CSRC.glob("*.h")]):
        for text in re.findall(r'asm volatile\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', src.read_text()):
            ops = [o.split()[0:2] for o in re.sub(r'"\s*"', "", text).strip().strip('"').replace("\\t", "").split("\\n")]
            for a, b in zip(ops, ops[1:]):
                assert not (a[1:2] == ["m0,"] and "lds" in b[0]), f"{src.name}: {text}"
            found += any("lds" in o[0] for o in ops)
    assert found >= 3
