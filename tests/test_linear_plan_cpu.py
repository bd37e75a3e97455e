"""The projections' dispatch rules (tgohip_linear_plan, host arithmetic) swept over forms,
activations, widths and rows: every call the allocation-free linear takes fits its array."""
import os
import subprocess
import sys

import pytest

import tgo_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

ARRAY = 64 << 20
WIDTHS = [(64, 128), (320, 6144), (1024, 6144), (1024, 65536), (1024, 151936), (1600, 34816), (1600, 49152),
          (2048, 1024), (2048, 32768), (4096, 4096), (4096, 24576), (4096, 151936), (5120, 51200), (5504, 32768),
          (12288, 4096), (25600, 5120)]
ROWS = sorted(set(list(range(1, 200)) + list(range(200, 1400, 37)) + [383, 384, 385, 2048, 2100, 4200]))


def plane_bytes(M, N):
    page = 2 << 20
    return -(-M * N * 4 // page) * page


@pytest.mark.parametrize("xd", [tgo_amd.F32, tgo_amd.F16, tgo_amd.F16X2])
@pytest.mark.parametrize("form", [0, 1, 2, 3])
def test_what_the_static_array_takes_fits_it(form, xd):
    """A call whose limit is at most 64 MiB runs: its planes fit the array, or it is the
    pipelined kernel's, which goes in bands of rows."""
    banded = 0
    for K, N in WIDTHS:
        for M in ROWS:
            p = tgo_amd.linear_plan(form, K, N, xd, M)
            if p.limit_bytes > ARRAY:
                continue
            at = (form, K, N, xd, M, p.kernel, p.splits)
            whole = p.splits * plane_bytes(M, N) if p.splits > 1 else 0
            assert p.array_bytes <= ARRAY, at
            assert whole <= ARRAY or p.kernel == tgo_amd.LINEAR_PIPE, at
            assert p.splits == 1 or p.array_bytes > 0, at
            banded += whole > ARRAY
    assert banded or xd == tgo_amd.F16, "the widths reach calls whose planes go in bands"


@pytest.mark.parametrize("most", [None, 1, 2, 4, 8])
def test_max_splits_bounds_every_pipelined_call(most):
    """TGOHIP_GEMM_MAX_SPLITS (read once per process) is the most split-K slices of the
    pipelined kernel, in both arithmetics; unset, 8, and 16 with activation pairs."""
    code = """
import tgo_amd
most = {}
for form in range(4):
    for xd in (tgo_amd.F32, tgo_amd.F16, tgo_amd.F16X2):
        for K, N in [(1024, 6144), (1600, 4096), (4096, 4096), (4096, 6144), (12288, 4096), (25600, 5120)]:
            for M in list(range(33, 200)) + [256, 353, 512, 1152, 1353]:
                p = tgo_amd.linear_plan(form, K, N, xd, M)
                if p.kernel == tgo_amd.LINEAR_PIPE:
                    most[xd] = max(most.get(xd, 0), p.splits)
print(most[tgo_amd.F32], most[tgo_amd.F16], most[tgo_amd.F16X2])
"""
    env = {k: v for k, v in os.environ.items() if not k.startswith("TGOHIP_")}
    if most:
        env["TGOHIP_GEMM_MAX_SPLITS"] = str(most)
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, capture_output=True, text=True, check=True)
    assert out.stdout.split() == ([str(most)] * 3 if most else ["16", "8", "16"])


@pytest.mark.parametrize("form", [0, 1, 2, 3])
def test_the_row_kernel_gets_only_calls_that_it_has(form):
    """It stores a SwiGLU (gate and up side by side: two column blocks a workgroup) as f16 or as
    a pair, not as f32, and pairs column blocks over more than 32 rows for f16 weights with f16
    rows or pairs only. Every combination of activation and epilogue that a call may have."""
    rows = 0
    for xd in (tgo_amd.F32, tgo_amd.F16, tgo_amd.F16X2):
        for epi in ((0, 1, 2, 5) if xd == tgo_amd.F16X2 else (0, 1, 2, 3, 4)):
            for K, N in WIDTHS:
                for M in ROWS:
                    p = tgo_amd.linear_plan(form, K, N, xd, M, epi)
                    if p.kernel != tgo_amd.LINEAR_ROWS:
                        continue
                    rows += 1
                    at = (form, K, N, xd, M, epi, p.column_blocks)
                    assert epi != 4, at
                    assert p.column_blocks == 2 or epi not in (3, 5), at
                    assert p.column_blocks == 1 or M <= 32 or (form == tgo_amd.FORM_F16 and xd != tgo_amd.F32), at
    assert rows > 1000
