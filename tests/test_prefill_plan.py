"""The 16-bit prefill's choice of kernel (plan_mfma, csrc/prefill.hip), asked through the plan query on
the CPU, where it plans for 256 CUs: what it reports is a form that exists, every grid fits a launch,
and asking costs little, since every call asks."""
import ctypes
import math
import random
import time

import pytest

import cdna4

# (kernel, waves, rows) of every form, by head dimension
FORMS = {
    64: {("fa_mfma_8w", 8, 256), ("fa_mfma_keys", 8, 128), ("fa_mfma_keys", 8, 64), ("fa_mfma_keys", 8, 32),
         ("fa_mfma_4w", 4, 64), ("fa_small", 8, 16), ("fa_small", 4, 16)},
    128: {("fa_mfma_8w", 8, 256), ("fa_mfma_keys", 8, 128), ("fa_mfma_keys", 8, 64), ("fa_mfma_4w", 4, 64),
          ("fa_small", 4, 16), ("fa_small", 2, 16)},
}


def plan(D, SQ, SK, HQ, HK, B, causal, dtype=cdna4.BF16):
    return cdna4.prefill_plan(cdna4.PrefillCfg(D, SQ, SK, HQ, HK, B, causal), dtype)


def shapes(count, seed):
    rng = random.Random(seed)

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    for _ in range(count):
        causal = rng.choice([0, 1])
        SQ = log_int(1, 9000)
        HK = rng.choice([1, 2, 3, 8, 12, 17, 32])
        yield (rng.choice([64, 128]), SQ, SQ if causal else log_int(1, 9000), HK * rng.choice([1, 2, 4, 8]), HK,
               log_int(1, 200), causal), rng.choice([cdna4.F16, cdna4.BF16])


def test_the_reported_kernel_is_the_form_that_runs():
    seen = {64: set(), 128: set()}
    for c, dt in shapes(6000, 1):
        p = plan(*c, dt)
        form = (p.name, p.waves, p.rows)
        assert form in FORMS[c[0]], (c, form)
        items = c[5] * c[3] * -(-c[1] // p.rows)
        assert p.grid == (min(items, 256) if p.rows == 256 else items), (c, form, p.grid)
        seen[c[0]].add(form)
    assert seen == FORMS   # and every form is chosen somewhere


@pytest.mark.parametrize("c", [(64, 1, 1, 128, 128, 131072, 0), (128, 1, 1, 128, 128, 262144, 0),
                               (64, 1, 1, 64, 64, 131071, 1), (64, 17, 17, 64, 64, 131072, 1),
                               (128, 3, 70, 64, 8, 400000, 0), (64, 64, 64, 1, 1, 16777216, 1),
                               (128, 129, 129, 8, 8, 2097152, 1)])
def test_grids_fit_a_launch(c):
    # fewer than 2^32 threads: what the one-workgroup-per-item forms cannot launch stays with the
    # persistent grid
    for dt in (cdna4.F16, cdna4.BF16):
        p = plan(*c, dt)
        assert p.grid * 64 * p.waves < 2 ** 32, (c, p.name, p.grid)


@pytest.mark.parametrize("c", [(128, 144, 144, 64, 16, 3, 1), (128, 247, 247, 32, 32, 6, 1), (128, 165, 165, 6, 3, 42, 1),
                               (128, 316, 316, 16, 4, 7, 1)])
def test_many_short_causal_sequences_take_four_waves_at_d128(c):
    # measured (us): the key-split forms 18.3, 23.4, 22.4, 22.2, fa_mfma 11.8, 19.9, 16.2, 16.6
    for dt in (cdna4.F16, cdna4.BF16):
        assert (plan(*c, dt).rows, plan(*c, dt).waves) == (64, 4)


def test_planning_costs_little_at_every_size():
    # Every call plans, so no shape may cost many times a small one's microsecond (a walk over all
    # items had taken 45-200 us at the sizes below).
    l, info = cdna4.lib(), cdna4.PlanInfo()

    def cost(c):
        cfg = cdna4.PrefillCfg(*c)
        args = (ctypes.byref(cfg), cdna4.BF16, ctypes.byref(info))
        best = 1e9
        for _ in range(20):
            t = time.perf_counter()
            for _ in range(20):
                l.cdna3_attn_prefill_plan(*args)
            best = min(best, (time.perf_counter() - t) / 20)
        return best

    small = cost((64, 64, 64, 8, 8, 1, 1))
    for c in [(128, 8192, 8192, 32, 32, 4, 1), (128, 2048, 2048, 32, 32, 100, 1), (128, 2048, 2048, 25, 25, 151, 1),
              (64, 16, 16, 12, 12, 2000, 1), (64, 512, 512, 8, 8, 2000, 1), (128, 2048, 2048, 17, 17, 240, 1),
              (128, 1700, 1700, 17, 17, 3, 1)]:
        assert cost(c) < 8 * small, (c, cost(c), small)
