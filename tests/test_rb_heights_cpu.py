"""The register-B GEMM's plan at any tile height (csrc/gemm_rbm.hip): the row tiles cover the rows with
no idle tile, no K range is empty, and the split-K planes fit the workspace the library asks for."""
import pytest

from infinitemodel_amd import _lib


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("cus", [256, 80])
def test_plans_cover_and_fit(bits, cus):
    taken = 0
    for N, K in [(4096, 14336), (28672, 4096), (6144, 4096), (4096, 4096), (2944, 768), (37, 64), (1000, 8192), (151936, 3584)]:
        for M in list(range(65, 130)) + [200, 255, 256, 257, 384, 511, 512, 513, 600, 777, 1024, 1850, 2048, 4096, 8192]:
            p = _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, 0 if bits == 8 else 64, N, sqn=K * bits // 8, cus=cus)
            if M > 512:
                assert p is not None
            if p is None:
                continue
            taken += 1
            ib, s = p[:2]
            rt = -(-M // (32 * ib))
            assert 3 <= ib <= 8 and (rt - 1) * 32 * ib < M
            kps = -(-(K // 64) // s)
            assert (s - 1) * kps < K // 64
            if s > 1:
                assert 4 * s * M * N <= 64 << 20
                if cus == 256:      # the query's device default when no GPU is there
                    assert _lib.lib().imq_linear_workspace_bytes(M, N, K) >= 4 * s * M * N
    assert taken > 100


def test_short_k_ranges_decline():
    """Few K steps a range and tiles past the CUs, or (up to 512 rows) a tile's fixed cost alone: the LDS-dequant GEMM's,
    measured. int4 and int8 stay above 512 rows, and a model's prefill shapes keep their plans."""
    plan = lambda b, M, N, K: _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, 0 if b == 8 else 64, N, sqn=K * b // 8)   # noqa: E731
    for M, N, K in ((200, 152064, 64), (512, 100000, 448), (256, 152064, 256)):
        assert all(plan(b, M, N, K) is None for b in (2, 4)), (M, N, K)
    assert plan(8, 96, 4096, 1024) is None and plan(8, 128, 2560, 2944) is None and plan(8, 150, 1008, 1024) is not None
    assert plan(2, 1024, 152064, 64) is None and plan(2, 1024, 40000, 512) is None and plan(2, 1024, 40000, 2048) is not None
    assert plan(4, 1024, 152064, 64) is not None and plan(8, 1024, 152064, 64) is not None
    for b in (2, 4, 8):
        for M, N, K in ((300, 28672, 4096), (384, 28672, 4096), (777, 28672, 8192), (2048, 4096, 14336)):
            assert plan(b, M, N, K) is not None, (b, M, N, K)
    assert plan(4, 200, 28672, 4096)[:2] == (7, 2) and plan(8, 512, 14336, 4096)[:2] == (4, 1) and plan(8, 512, 4096, 14336)[:2] == (4, 4)


def test_few_columns_of_int2_and_short_k_of_int8_decline():
    """Where the LDS-dequant GEMM measured faster; int4 of those columns, int2 of longer K and int8 past them stay."""
    plan = lambda b, M, N, K: _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, 0 if b == 8 else 64, N, sqn=K * b // 8)   # noqa: E731
    assert all(plan(2, M, 1024, 2048) is None and plan(4, M, 1024, 2048) is not None for M in (872, 985, 1170))
    assert plan(2, 985, 1024, 8192) is not None and plan(2, 985, 2048, 4096) is not None
    assert plan(8, 132, 12352, 192) is None and plan(8, 79, 256, 896) is None
    assert plan(8, 256, 14336, 640) is not None and plan(8, 200, 14336, 1024) is not None


def test_rows_up_to_64_and_odd_k_decline():
    assert _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, 64, 4096, 128, 4096, sqn=2048) is None
    assert _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, 600, 4096 + 32, 128, 4096, sqn=2064) is None


def test_the_two_height_planes_are_other_dtypes_need():
    """bf16 and fp16 scale and zero alike are the any-height GEMM's above 512 rows: the two-height GEMM's planes are not in
    such an int4 call's workspace."""
    f = _lib.lib().imq_linear_w4_workspace_bytes
    less = 0
    for M, N, K in ((513, 4096, 14336), (600, 1000, 14336), (600, 512, 4096), (1024, 1024, 28672), (2048, 4096, 14336), (2048, 4096, 4096), (900, 8192, 2048)):
        rb = _lib.launch_plan(_lib.IMQ_PLAN_GEMM_RB, M, K, 128, N, sdt=_lib.IMQ_DT_FP32)
        rbm = [_lib.launch_plan(_lib.IMQ_PLAN_GEMM_RBM, M, K, G, N, sqn=K * b // 8) for b, G in ((4, 128), (8, 0))]
        lds = _lib.launch_plan(_lib.IMQ_PLAN_GEMM, M, K, 128, N)
        planes = lambda s: 4 * s * M * N if s > 1 else 0   # noqa: E731
        own = max([planes(lds[2])] + [planes(p[1]) for p in rbm if p])
        st = (K // 2, K, K // 128, 1)
        assert f(M, K, N, 128, *st, 0, K // 128, 1, 0) == f(M, K, N, 128, *st, 1, K // 128, 1, 1) == own
        for s, z in ((2, 2), (0, 1), (0, 2)):
            assert f(M, K, N, 128, *st, s, K // 128, 1, z) == max(own, planes(rb[1]))
        less += own < planes(rb[1])
    assert less


def test_no_build_switch_picks_the_step():
    """The folded form's step and the dequantizing one are not interchangeable (only step_fold folds a group's sums), so
    what a build may override in the kernel's header are the scheduler's VALU counts alone."""
    import os
    import re
    src = open(os.path.join(os.path.dirname(_lib.__file__), "csrc", "rb_kernel.h")).read()
    assert set(re.findall(r"#\s*if(?:ndef|def)?\s+(\w+)", src)) == {"RB_VALU_PER_MFMA_2", "RB_VALU_PER_MFMA_4", "RB_VALU_PER_MFMA_8"}
