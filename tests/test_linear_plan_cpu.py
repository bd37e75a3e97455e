"""The projections' dispatch rules (tgohip_linear_plan, host arithmetic) swept over forms,
activations, widths and rows: every call the allocation-free linear takes fits its array."""
import pytest

import tgo_amd

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
