"""The plan of products that leave slabs: forms that the launch takes, as many slabs as it says at most."""
import ctypes as C

import pytest

from cake_amd.ops import gemm as G


@pytest.mark.parametrize("M", [1, 2, 16, 17, 32, 33, 64, 65, 200, 400, 3000])
def test_forms(M):
    lib = G._lib()
    for N in (4, 132, 1024, 4096, 6144, 8192, 128256):
        for K in (8, 264, 512, 1032, 4096, 11008, 28672):
            k, c, p = C.c_int(-1), C.c_int(-1), C.c_int(-1)
            on = lib.cake_gemm_slab_plan(M, N, K, 1, 0, C.addressof(k), C.addressof(c), C.addressof(p))
            assert on or M > 64
            if not on:
                continue
            assert 1 <= p.value <= 16
            if k.value == 2:
                steps = -(-K // (64 if M > 16 else 128))
                assert M <= 64 and (p.value == 1 or steps // p.value >= (8 if M > 16 else 4))
            elif k.value == 1:
                assert M <= 32 and p.value == 1
            else:
                assert k.value == 0 and c.value not in G.FOUR_WAVE and p.value >= 2 and K // 64 // p.value >= 3
