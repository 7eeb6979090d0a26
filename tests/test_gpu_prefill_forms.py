"""The prefill forms whose workgroups split the keys over their waves (fa_mfma_keys, csrc/prefill.hip),
and the persistent form's item orders, against the oracle on sampled rows of sampled heads (bounds as
in test_gpu_kernel_paths.py). Lengths around the forms' query blocks (128, 64, 32) and key steps (64,
128, 256): one past, one short, fewer keys than a step, blocks whose last waves hold no query."""
import pytest
import torch

import cdna4
from test_gpu_kernel_paths import check_prefill

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


def _form(D, SQ, SK, HQ, HK, B, causal, dtype, rows, waves, heads, seed):
    p = cdna4.prefill_plan(cdna4.PrefillCfg(D, SQ, SK, HQ, HK, B, causal), dtype)
    name = p.name
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (p.rows, p.waves) == (rows, waves)
        name = {256: "fa_mfma_8w", 16: "fa_small"}.get(rows, "fa_mfma_4w" if waves == 4 else "fa_mfma_keys")
    check_prefill(D, SQ, SK, HQ, HK, B, causal, dtype, name, seed=seed, heads=heads)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("D,SQ,SK,HQ,HK,B,causal,rows", [
    (128, 1531, 1531, 32, 8, 1, 1, 128),
    (128, 1665, 1665, 16, 16, 2, 1, 128),      # 13 blocks and one query
    (128, 257, 6431, 64, 8, 1, 0, 128),        # cross attention, keys one short of a step
    (64, 1825, 1825, 16, 4, 2, 1, 128),
    (128, 785, 785, 8, 8, 1, 0, 64),
    (128, 1025, 1025, 8, 2, 1, 1, 64),
    (128, 123, 123, 32, 8, 4, 0, 64),          # fewer keys than a step
    (128, 933, 393, 8, 8, 2, 0, 64),
    (64, 1545, 1545, 8, 1, 1, 0, 64),
    (64, 943, 943, 12, 12, 2, 1, 64),          # heads not a multiple of 8
    (64, 513, 513, 12, 12, 1, 1, 32),
    (64, 959, 959, 2, 2, 3, 1, 32),
    (64, 511, 511, 8, 8, 2, 1, 32),
])
def test_keys_split_forms(D, SQ, SK, HQ, HK, B, causal, rows, dtype):
    heads = [(b, h) for b in range(B) for h in range(0, HQ, max(1, HQ // 4))]
    _form(D, SQ, SK, HQ, HK, B, causal, dtype, rows, 8, heads, SQ + SK)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("D,S,HQ,HK,B", [
    (64, 301, 32, 8, 6),
    (64, 65, 64, 64, 9),       # one query past a block, one key past a tile
    (64, 129, 17, 17, 15),     # heads not a multiple of 8
    (128, 144, 64, 16, 3),
    (128, 65, 64, 64, 5),
    (128, 129, 17, 17, 15),
    (128, 316, 16, 4, 7),
])
def test_four_wave_form(D, S, HQ, HK, B, dtype):
    _form(D, S, S, HQ, HK, B, 1, dtype, 64, 4, [(0, 0), (B // 2, HQ // 3), (B - 1, HQ - 1)], S + D)


@pytest.mark.parametrize("D,S,HQ,HK,B,causal", [
    (128, 2675, 8, 1, 7, 1),     # heaviest blocks of all heads first (uneven head-major rounds)
    (64, 2100, 40, 8, 3, 1),
    (128, 1700, 17, 17, 3, 1),   # heads not a multiple of 8: no XCD grouping, a partial odd round
    (128, 2060, 21, 21, 3, 0),
])
def test_persistent_item_orders(D, S, HQ, HK, B, causal):
    _form(D, S, S, HQ, HK, B, causal, BF16, 256, 8, [(0, 0), (0, HQ - 1), (B - 1, HQ // 2), (B - 1, HQ - 1)], S)
