"""CPU checks of the launch rules of five to sixteen rows (the planner is host code): where narrow projections run unsplit, with how
many waves, and how many K splits a K that does not fit LDS takes. Each line is where the measured times cross, on both sides."""

import collections
import ctypes

import pytest

from heteromega_amd import _lib

Plan = collections.namedtuple("Plan", "one_math strips groups splits nu wps units partial_bytes")


def gemv_plan(m, n, k, group, dtype, fused=False, cus=256):
    out = (ctypes.c_int64 * 8)()
    fn = ctypes.CDLL(_lib.LIB_PATH).hm_gemv_plan_of
    fn.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int32] * 3 + [ctypes.c_int64, ctypes.c_void_p]
    fn.restype = None
    fn(m, n, k // 128, group, {"bf16": _lib.HM_BF16, "fp16": _lib.HM_FP16}[dtype], int(fused), cus, out)
    return Plan(*out)


@pytest.mark.parametrize("m,n,k,group,dtype,unsplit", [
    # strip pairs of a long K: few of them stay split
    (16, 2048, 4224, 128, "fp16", False), (16, 2560, 4224, 128, "fp16", True), (16, 2048, 5120, 64, "fp16", False),
    (16, 2560, 5120, 64, "fp16", True), (12, 2048, 5120, 64, "fp16", True), (12, 1536, 5120, 64, "fp16", False), (9, 1024, 4608, 128, "fp16", False), (9, 1024, 4096, 128, "fp16", True),
    (8, 1024, 5120, 64, "fp16", False), (8, 1536, 5120, 64, "fp16", True), (9, 6144, 5248, 128, "fp16", False),
    (9, 6144, 4096, 128, "fp16", True), (9, 8256, 4096, 128, "fp16", False),
    # strip pairs in groups of 32
    (12, 4096, 4096, 32, "fp16", False), (12, 6144, 4096, 32, "fp16", True),
    # single strips
    (8, 512, 8192, 64, "bf16", True), (8, 1024, 7168, 64, "bf16", True), (8, 1024, 7680, 64, "bf16", False), (8, 1536, 8192, 64, "bf16", True),
    (8, 1536, 8320, 64, "bf16", False), (8, 512, 6144, 32, "bf16", True), (8, 512, 6656, 32, "bf16", False),
    (8, 1536, 8192, 32, "bf16", True)])
def test_narrow_projections(m, n, k, group, dtype, unsplit):
    p = gemv_plan(m, n, k, group, dtype)
    assert not p.one_math
    assert (p.splits == 1) == unsplit, p


@pytest.mark.parametrize("k,group,dtype,waves", [(1920, 64, "fp16", 4), (2048, 64, "fp16", 8), (2048, 32, "bf16", 8), (3968, 128, "fp16", 4),
                                                 (4096, 128, "fp16", 8)])
def test_waves_of_an_unsplit_projection(k, group, dtype, waves):
    p = gemv_plan(16, 2048, k, group, dtype)
    assert (p.splits, p.nu, p.wps) == (1, 1, waves), p


@pytest.mark.parametrize("group", [64, 128])
@pytest.mark.parametrize("m", [6, 9, 12, 16])
def test_long_k_takes_at_most_eight_splits(m, group):
    # more splits than the split sum loads at once were slower at these widths (narrower ones may take more by the first weights)
    for n in (2048, 2560, 3072, 4096, 5120, 8192):
        for k in range(6144, 16384, 1024):
            p = gemv_plan(m, n, k, group, "fp16")
            assert p.one_math or p.splits <= 8, (m, n, k, p)


def test_downs_at_sixteen_rows():
    # Llama-3-8B, Qwen2.5-14B and Llama-3.2-1B: the finer splits that their times were measured with
    assert gemv_plan(16, 4096, 14336, 128, "fp16").splits == 8
    assert gemv_plan(16, 5120, 13824, 64, "fp16").splits == 6
    assert gemv_plan(16, 2048, 8192, 128, "fp16").splits == 8
