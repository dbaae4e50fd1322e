"""The footprint covers the source table: a shot's box may hold up to 4096 points
(all of a smaller grid), 36 rates each.  Servers admit shots by this number."""
import ctypes as C

import pytest

import cgfd


@pytest.mark.parametrize("storage,es,ms", [(cgfd.STORE_F32, 4, 4), (cgfd.STORE_F16, 2, 4), (cgfd.STORE_BF16, 2, 4),
                                           (cgfd.STORE_F64, 8, 8)])
@pytest.mark.parametrize("n,cells", [(40, 4096), (12, 12 ** 3)])
def test_each_shot_counts_the_largest_source_table(n, cells, storage, es, ms):
    lib = cgfd.load()
    one, two = (lib.cgfd_footprint_bytes(C.byref(cgfd.Desc(n, n, n, storage, k, 0)), 0, 0) for k in (1, 2))
    align = 128 // es
    px = (align + n + 3 + align - 1) // align * align
    levels = 4 * 9 * px * (n + 6) * (n + 6) * es
    memory = 5 * 9 * (6 * 11 * n * n) * es   # PML memory of six 11-point faces
    maps = 18 * n * n * ms                   # peak ground motion
    assert two - one >= levels + memory + maps + 36 * cells * ms
