"""When launches split (csrc/split.h), through the queries of their scratch: on the CPU."""
import random

import pytest

from dmad_amd import _native as nat

BF16, F16, F32 = nat.DMAD_BF16, nat.DMAD_F16, nat.DMAD_F32
PLAIN, JVP, QONLY = nat.DMAD_FWD_PLAIN, nat.DMAD_FWD_JVP, nat.DMAD_FWD_JVP_KV_TANGENT_ZERO


def _sizes(seed, n):
    r = random.Random(seed)
    for _ in range(n):
        yield r.choice([1, 2, 4]), r.choice([1, 2, 5, 12, 40]), int(2 ** r.uniform(0, 20)), int(2 ** r.uniform(0, 20))


def test_partials_are_bounded():
    for B, H, Lq, Lk in _sizes(1, 400):
        for D in (16, 64, 128, 256):
            for dt in (BF16, F32):
                assert 0 <= nat.fwd_split_bytes(dt, PLAIN, B, H, Lq, Lk, D, D) <= 128 << 20
                assert 0 <= nat.fwd_split_bytes(dt, JVP, B, H, Lq, Lk, D, D) <= 128 << 20
            assert 0 <= nat.bwd_split_bytes(BF16, False, False, B, H, Lq, Lk, D) <= 128 << 20
            if D <= 128:
                assert 0 <= nat.bwd_split_bytes(F16, True, True, B, H, Lq, Lk, D) <= 128 << 20
        assert 0 <= nat.magi_split_bytes(BF16, (Lq + 127) // 128, (Lk + 31) // 32, B, H, 128, 128) <= 128 << 20


def test_jvp_modes_split_alike():
    """O must not depend on whether Kd = Vd = 0 was stated."""
    some = 0
    for B, H, Lq, Lk in _sizes(2, 400):
        for dt in (BF16, F16, F32):
            for D in (64, 128):
                a, b = (nat.fwd_split_bytes(dt, m, B, H, Lq, Lk, D, D) for m in (JVP, QONLY))
                assert a == b, (dt, B, H, Lq, Lk, D)
                some += a > 0
    assert some > 50
    # the short key ranges of the two-workgroups-per-CU kernel: none up to 512 keys, and up to 2048
    # only where CUs would have no tile at all
    assert nat.fwd_split_bytes(BF16, QONLY, 1, 1, 4000, 512, 128, 128) == 0
    assert nat.fwd_split_bytes(BF16, QONLY, 1, 10, 3300, 2048, 128, 128) == 0
    assert nat.fwd_split_bytes(BF16, QONLY, 1, 2, 700, 2048, 128, 128) > 0


def test_full_rounds_and_other_head_dims_stay_whole():
    for mode in (PLAIN, JVP, QONLY):
        assert nat.fwd_split_bytes(BF16, mode, 1, 40, 32760, 32760, 128, 128) == 0  # 40 rounds of 256 tiles
        for D in (16, 32, 256):
            assert nat.fwd_split_bytes(BF16, mode, 1, 2, 3000, 9000, D, D) == 0
        assert nat.fwd_split_bytes(F32, mode, 1, 2, 3000, 9000, 64, 128) == 0
    assert nat.bwd_split_bytes(BF16, False, False, 1, 40, 32760, 32760, 128) == 0
    assert nat.bwd_split_bytes(F32, False, False, 1, 2, 3000, 3000, 128) == 0
    assert nat.magi_split_bytes(BF16, 40, 0, 1, 2, 128, 128) == 0  # a mask that does not say how long its tasks are


@pytest.mark.parametrize("L,pieces", [(1560, 2), (1731, 3), (1800, 2)])
def test_pieces_fit_the_engines(L, pieces):
    """Workgroups go to an XCD's four engines in turn: 168 tiles (1731 tokens) in uneven pairs would
    leave one engine six long and five short pieces, as long as the whole tiles."""
    tiles, part = (L + 127) // 128 * 12, 4 * (2 * 128 * 128 + 3 * 128)  # O, C and three statistics of 128 rows
    assert nat.fwd_split_bytes(F32, JVP, 1, 12, L, L, 128, 128) == tiles * pieces * part


@pytest.mark.parametrize("D,slots", [(64, 512), (128, 256)])
def test_masks_split_where_their_tasks_fit_the_chip_or_belong_to_few_heads(D, slots):
    """Tasks differ in length: with whole tasks in the launch a cut slows most masks of four and more
    heads down, and those of fewer heads where hardly any task is left to cut; walks of 24 tiles are
    over before the host has issued two launches."""
    for BH in (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 20, 24, 40):
        for tasks in range(1, 4 * slots // BH + 2):
            items, rest = tasks * BH, tasks * BH % slots
            for kt in (24, 60, 200, 500):
                if kt == 24 or (items > slots and (BH > 3 or rest < slots // 32)):
                    assert nat.magi_split_bytes(BF16, tasks, kt, 1, BH, D, D) == 0, (BH, tasks, kt)
    assert nat.magi_split_bytes(BF16, slots // 4, 200, 1, 1, D, D) > 0
    assert nat.magi_split_bytes(BF16, slots // 128, 200, 2, 12, D, D) > 0
    assert nat.magi_split_bytes(BF16, slots // 3 + 7, 200, 3, 1, D, D) > 0


def test_argument_checks():
    with pytest.raises(ValueError):
        nat.fwd_split_bytes(BF16, JVP, 1, 2, 64, 64, 96, 96)
    with pytest.raises(ValueError):
        nat.fwd_split_bytes(BF16, 7, 1, 2, 64, 64, 64, 64)
    with pytest.raises(ValueError):
        nat.bwd_split_bytes(BF16, False, False, -1, 2, 64, 64, 64)
    with pytest.raises(ValueError):
        nat.magi_split_bytes(BF16, 4, -1, 1, 2, 64, 64)
