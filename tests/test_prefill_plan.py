"""The 16-bit prefill's choice of kernel (plan_mfma, csrc/prefill.hip), asked through the plan query on
the CPU, where it plans for 256 CUs."""
import pytest

import cdna4


def plan(D, SQ, SK, HQ, HK, B, causal, dtype=cdna4.BF16):
    return cdna4.prefill_plan(cdna4.PrefillCfg(D, SQ, SK, HQ, HK, B, causal), dtype)


@pytest.mark.parametrize("c", [(128, 144, 144, 64, 16, 3, 1), (128, 247, 247, 32, 32, 6, 1), (128, 165, 165, 6, 3, 42, 1),
                               (128, 316, 316, 16, 4, 7, 1)])
def test_many_short_causal_sequences_take_four_waves_at_d128(c):
    # measured (us): the key-split forms 18.3, 23.4, 22.4, 22.2, fa_mfma 11.8, 19.9, 16.2, 16.6
    for dt in (cdna4.F16, cdna4.BF16):
        assert (plan(*c, dt).rows, plan(*c, dt).waves) == (64, 4)
