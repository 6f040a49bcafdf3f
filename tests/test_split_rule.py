"""The split rules (va_pick_splits, va_pick_splits_gqa): whole rounds of work-groups where
heads do not divide the CUs, and decodes at such counts on the GPU."""
import numpy as np
import pytest

import oracle
import voltattn_amd as va
from oracle import batch
from tests import gpu_util
from tests.numerics import cond_bound

TILED = [va.Fmt.F16M, va.Fmt.Q8M, va.Fmt.Q4M, va.Fmt.Q3M]
CUS = 256          # without a GPU, and on MI355X


@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("L", [1, 4097, 10007, 262144])
def test_groups_fit_whole_rounds(fmt, L):
    two = fmt in (va.Fmt.Q8M, va.Fmt.Q4M)
    for H in range(1, 256):
        S = va.pick_splits(fmt, H, L, 128)
        rounds = 2 if two and H * (CUS // H) < CUS - CUS // 32 and H * L >= 1280 * CUS else 1
        if H > CUS // 2 and rounds == 1:        # rounded up: down would idle up to half the CUs
            assert 1 <= S <= 2, (H, S)
            continue
        assert 1 <= S and H * S <= rounds * CUS, (H, S)
        assert (S - 1) * va.split_chunk(L, S) < L, (H, S)            # no split is empty
    for Hkv in (1, 5, 6, 10, 12, 48, 100):
        assert Hkv * va.pick_splits_gqa(fmt, 4 * Hkv, Hkv, L, 128) <= CUS


@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("B,Hq,Hkv", [(2, 32, 8), (16, 8, 8), (64, 32, 8), (100, 64, 8)])
@pytest.mark.parametrize("L", [300, 16384, 1 << 20])
def test_paged_splits_hold_pieces_and_pages(fmt, B, Hq, Hkv, L):
    """The picked count keeps a split, in whole kernel tiles (512 positions at most), within
    the pages that a work-group stages (1024), for calls that get no ticket slot, as well as
    giving the workspace of a balanced launch: a partial per merge group and per work-group."""
    shape = va.PagedShape(B, Hq, Hkv, 128, 32, 64, L // 64 + 1, 1 << 14, L)
    S = va.pick_splits_paged(fmt, shape)
    chunk = -(-(-(-L // 512)) // S) * 512
    assert S >= 1 and chunk // 64 + 2 <= 1024, S
    qg = min(4, Hq // Hkv)
    groups = B * Hq // qg
    if L < 1 << 20 and groups <= 1024 and (groups > CUS or groups * L >= 2048 * CUS):
        assert B * Hq * S // qg >= groups + CUS, S


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("H,L", [(33, 10300), (40, 8191), (60, 2000)])
def test_odd_head_counts(fmt, H, L):
    c = gpu_util.case(va.fmt_bits(fmt), H, L, 64, 32, 0x0DD + H)
    S = va.pick_splits(fmt, H, L, 64)
    print(f"odd heads {fmt.label} H={H} L={L} S={S}", flush=True)
    got = np.asarray(gpu_util.run_case(fmt, c, S)["out"], np.float64).ravel()
    ref = np.asarray(c["ref"], np.float64).ravel()
    mag = np.asarray(batch.magnitude_gqa(c["kd"], c["vd"], c["q"], H, H, L, 64)).ravel()
    assert oracle.gate(got, ref)[0]
    assert np.all(np.abs(got - ref) <= cond_bound(ref, mag))
