"""fp32 prefill (fa_f32) with one and two query tiles per workgroup against fp64: ragged query and key
counts, grouped-query heads, causal and not, an output that starts at an odd float, and the edge of
the rule that takes two tiles."""
import math

import pytest
import torch

import cdna4
from gpu_util import DEV

pytestmark = pytest.mark.gpu


def reference(Q, K, V, causal):
    B, HQ, SQ, D = Q.shape
    rep = HQ // K.shape[1]
    q, k, v = (t.double().reshape(-1, t.shape[2], D) for t in (Q, K.repeat_interleave(rep, 1), V.repeat_interleave(rep, 1)))
    out = []
    for i in range(B * HQ):
        s = q[i] @ k[i].t().contiguous() / math.sqrt(D)
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
        out.append(torch.softmax(s, 1) @ v[i])
    return torch.stack(out).reshape(B, HQ, SQ, D)


@pytest.mark.parametrize("B,HQ,HK,SQ,SK,D,causal,rows", [
    (1, 1, 1, 1, 1, 64, 0, 16), (2, 3, 1, 15, 131, 64, 0, 16), (1, 8, 2, 129, 129, 64, 1, 16),
    (1, 2, 2, 17, 15, 128, 0, 16), (1, 4, 1, 255, 255, 128, 1, 16), (3, 8, 8, 1001, 77, 64, 0, 16),
    (2, 12, 4, 1021, 1021, 128, 1, 32), (2, 12, 12, 993, 129, 128, 0, 32), (96, 8, 2, 3, 17, 128, 0, 32),
    (48, 16, 16, 33, 33, 128, 1, 32), (2, 12, 4, 992, 40, 128, 0, 16),
])
def test_f32_tiles(B, HQ, HK, SQ, SK, D, causal, rows):
    g = torch.Generator(device=DEV).manual_seed(SQ * 7 + SK)
    Q, K, V = (torch.randn(B, h, s, D, generator=g, device=DEV) for h, s in ((HQ, SQ), (HK, SK), (HK, SK)))
    cfg = cdna4.PrefillCfg(D, SQ, SK, HQ, HK, B, causal)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        plan = cdna4.prefill_plan(cfg, cdna4.F32)
        assert plan.name == "fa_f32" and plan.rows == rows and plan.grid == B * HQ * -(-SQ // rows)
    buf = torch.full((Q.numel() + 9,), 55.0, device=DEV)
    O = buf[1:1 + Q.numel()].view(Q.shape)
    cdna4.prefill(Q, K, V, O, cfg)
    # Chains of at most SK / 8 products per wave (plus the merge) and of D products per score, scores
    # of order one: eps per step, on values up to max|V|.
    tol = 2.0 ** -24 * (SK / 8 + 2 * D) * float(V.abs().max())
    err = float((O.double() - reference(Q, K, V, causal)).abs().max())
    assert err <= tol, (err, tol)
    assert buf[0] == 55.0 and (buf[1 + Q.numel():] == 55.0).all()
