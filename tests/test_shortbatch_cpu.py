"""The short-batch GEMM's plan and address arithmetic (csrc/gemm_wk.h), restated: every K step is taken by
one wave of one range, every operand read lies inside its buffer, the line-tiled offsets are the
layout's definition, the staged scale groups cover the steps that use them, and the LDS regions fit."""
import ctypes

import numpy as np
import pytest

from infinitemodel_amd import _lib
from tests import _cases as C

WAVES, BK = 8, 64


def _plan(bits, M, N, K, G, cus=256, lds=160 * 1024):
    got = _lib.launch_plan(_lib.IMQ_PLAN_GEMM_WK, M, K, G, N, sqn=K * bits // 8, max_lds=lds, cus=cus)
    return got and got[:2]


def _szs(jb):
    return 32 * jb + {1: 4, 2: 8, 4: 16}[jb]


CASES = [(4, 17, 28672, 4096, 128), (4, 64, 28672, 4096, 128), (4, 32, 4096, 14336, 128), (4, 20, 37, 64, 64),
         (4, 33, 1008, 448, 32), (2, 64, 8192, 28672, 64), (2, 17, 96, 448, 64), (8, 40, 4096, 14336, 0),
         (8, 17, 40, 64, 0), (8, 5, 4096, 14336, 0), (8, 16, 152064, 3584, 0), (4, 24, 256, 8192, 128), (4, 17, 151936, 3584, 128)]


@pytest.mark.parametrize("bits,M,N,K,G", CASES)
@pytest.mark.parametrize("cus,lds", [(256, 160 * 1024), (32, 64 * 1024)])
def test_plan_and_addresses(bits, M, N, K, G, cus, lds):
    p = _plan(bits, M, N, K, G, cus, lds)
    if p is None:
        assert lds < 160 * 1024          # only a small LDS refuses a shape
        return
    jb, splits = p
    ib, KT_all = (1 if M <= 32 else 2), K // BK
    kps = -(-KT_all // splits)
    rj = 2 if ib == 1 and jb > 1 else 1
    gsh = G.bit_length() - 1 if G else 0
    groups_alloc = 0 if bits == 8 else ((kps * BK) >> gsh) + 2
    region = WAVES * ib * rj * 4096
    assert region + groups_alloc * _szs(jb) * 4 <= lds
    taken = np.zeros(KT_all, int)
    for split in range(splits):
        kt0 = split * kps
        KT = min(KT_all - kt0, kps)
        assert KT >= 1
        g_lo, g_hi = (kt0 * BK) >> gsh, ((kt0 + KT) * BK - 1) >> gsh
        assert bits == 8 or g_hi - g_lo + 1 <= groups_alloc
        for wave in range(WAVES):
            steps = (KT - wave + WAVES - 1) // WAVES if KT > wave else 0
            for i in range(steps + 2):                       # loads run up to two steps ahead, clamped
                kt = kt0 + min(wave, KT - 1) + WAVES * max(min(i, steps - 1), 0)
                assert kt0 <= kt < kt0 + KT
                if i < steps:
                    taken[kt] += 1
                    if bits != 8:
                        for h in range(2):
                            assert g_lo <= (kt * BK + 32 * h) >> gsh <= g_hi
    assert (taken == 1).all()
    # activation rows and chunks of a step: 32 ib rows of 8 chunks, each LDS slot once
    slots = set()
    for j in range(4 * ib):
        for lane in range(64):
            row, ch = 8 * j + (lane >> 3), lane & 7
            slots.add((row * 8 + (ch ^ ((row >> 1) & 7))) * 16)
            assert min(row, M - 1) * K + ch * 8 + (KT_all - 1) * BK + 8 <= M * K
    assert slots == set(range(0, ib * 4096, 16))
    # the sums' quads fill the same regions
    assert max(((u * ib + b) * 4 + r4) * 64 + lane for u in range(rj) for b in range(ib) for r4 in range(4)
               for lane in (63,)) * 16 + 16 == ib * rj * 4096


@pytest.mark.parametrize("bits,K", [(4, 512), (2, 1024), (8, 256)])
def test_tiled_offsets_are_the_layout(bits, K):
    """Lane (column c, half h) at K step kt reads, at its tiled offset, the bytes [QB (2 kt + h), + QB) of
    its row (QB = 4 bits), int8 in two 16-byte pieces 256 bytes apart."""
    N = 48
    q = np.random.default_rng(bits).integers(0, 256, (N, K * bits // 8), dtype=np.uint8)
    flat, sqn, QB = C.line_tile_np(q).reshape(-1), K * bits // 8, 4 * bits
    for rr in range(N):
        for h in range(2):
            hr = (rr >> 3) & 1
            qo = (rr >> 4) * 16 * sqn + 1152 * hr + 16 * (rr & 7) + {8: 512, 4: 256, 2: 8}[bits] * h
            for kt in range(K // BK):
                sel = {8: kt, 4: kt >> 1, 2: kt >> 2}[bits] & 1
                so = {8: 2048 * (kt >> 1), 4: 2048 * (kt >> 2) + 512 * (kt & 1),
                      2: 2048 * (kt >> 3) + 256 * (kt & 3)}[bits]
                at = (qo ^ (sel << 7)) + so
                got = np.concatenate([flat[at + 256 * v: at + 256 * v + min(QB, 16)] for v in range(2 if bits == 8 else 1)])
                assert np.array_equal(got, q[rr, QB * (2 * kt + h): QB * (2 * kt + h) + QB])


def test_small_devices_and_other_rows_decline():
    assert _plan(4, 16, 4096, 4096, 128) is None and _plan(4, 65, 4096, 4096, 128) is None
    assert _plan(4, 17, 4096, 4096 + 32, 128) is None
    assert _plan(8, 4, 4096, 4096, 0) is None and _plan(8, 5, 4096, 4096, 0) is not None      # int8 from 5 rows
    assert _plan(8, 8, 65552, 4096, 0) is None and _plan(8, 9, 65552, 4096, 0) is not None


@pytest.mark.parametrize("bits", [2, 4, 8])
def test_every_splitting_plan_fits_the_workspace_bound(bits):
    """The bytes the library asks for hold every plan's planes at the library's own default of 256 CUs (int8 from 5
    rows, K of any multiple of 64: with too few bytes the call would run unsplit)."""
    split = 0
    for K in (64, 1088, 1152, 2112, 3520, 4096, 6784, 8192, 10368, 13696, 14336, 28672):
        for N in (37, 512, 1024, 2688, 4096, 6208, 14336, 65536):
            for M in (5, 8, 9, 12, 14, 16, 17, 24, 32, 33, 48, 64):
                p = _plan(bits, M, N, K, 0 if bits == 8 else 64)
                if p is None or p[1] == 1:
                    continue
                split += 1
                assert 4 * p[1] * M * N <= _lib.lib().imq_linear_workspace_bytes(M, N, K), (M, N, K, p)
    assert split > (200 if bits == 8 else 100)


def test_short_k_and_wide_n_decline():
    """Where the workgroups outnumber the CUs and each has few K steps, the LDS-dequant GEMM (int8 decode rows: the skinny
    kernel) measured faster; at a model's widths the form keeps its rows."""
    for bits in (2, 4, 8):
        G = 0 if bits == 8 else 64
        for M in (17, 33, 64):
            assert _plan(bits, M, 131072, 64, G) is None and _plan(bits, M, 4096, 64, G) is not None
            for N, K in ((4096, 4096), (6144, 4096), (28672, 4096), (4096, 14336), (14336, 4096), (8192, 28672), (152064, 3584), (9728, 896)):
                assert _plan(bits, M, N, K, G) is not None, (bits, M, N, K)
        assert _plan(bits, 64, 65536, 512, G) is None and _plan(bits, 64, 65536, 2048, G) is not None
    assert _plan(8, 8, 65536, 192, 0) is None and _plan(8, 9, 65536, 192, 0) is not None
    assert _plan(8, 16, 20000, 64, 0) is None and _plan(8, 16, 16384, 64, 0) is not None


def test_int8_rows_5_to_8_just_past_the_cus_decline():
    """A second, nearly empty round of workgroups: the skinny kernel's, while it can stage the rows."""
    for M in (5, 6, 8):
        assert _plan(8, M, 18944, 3584, 0) is None and _plan(8, M, 16384, 3584, 0) is not None
        assert _plan(8, M, 28672, 4096, 0) is not None and _plan(8, M, 18944, 14336, 0) is not None
    assert _plan(8, 9, 18944, 3584, 0) is not None and _plan(8, 8, 18944, 512, 0) is not None


@pytest.mark.parametrize("bits,M", [(4, 17), (4, 32), (4, 64), (4, 200), (4, 1024), (2, 17), (2, 64), (2, 1024)])
@pytest.mark.parametrize("dts", [(0, 1), (0, 2), (1, 0), (2, 0)])
def test_line_tiled_weights_of_mixed_dtypes_are_refused(bits, M, dts):
    """Past 16 rows a line-tiled call's scale and zero have one dtype, whichever GEMM would take its row count. Refused
    before any launch: the pointers are never read."""
    L, K, N, G = _lib.lib(), 1024, 64, 128 if bits == 4 else 64
    p = ctypes.c_void_p(1 << 20)
    rc = (L.imq_linear_w4_tiled if bits == 4 else L.imq_linear_w2_tiled)(
        p, K, M, K, p, K * bits // 8, p, K // G, 1, dts[0], p, K // G, 1, dts[1], N, G, p, N, None, 0, None)
    assert rc == _lib.IMQ_ERR_UNSUPPORTED
