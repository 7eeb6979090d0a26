"""Session norms with and without a bias: bias files that hold zeros give exactly the logits and tokens
of none at all, for RMSNorm and LayerNorm, in the prompt and in the decode steps."""
import os

import numpy as np
import pytest

import cdna4
from cdna4 import model_format

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norm", ["rms", "layernorm"])
def test_zero_norm_bias_equals_none(tmp_path, norm):
    d = str(tmp_path)
    model_format.random_model(d, n_layers=2, hidden=192, n_heads=3, ffn_dim=320, vocab_size=501, norm=norm, seed=3)
    names = ["final_norm_bias"] + [f"layer_{i}_norm_{k}_bias" for i in range(2) for k in ("attn", "mlp")]
    outs = []
    for present in (True, False):
        for name in names:
            f = os.path.join(d, name + ".bin")
            if present:
                np.zeros(192, dtype="<f2").tofile(f)
            elif os.path.exists(f):
                os.remove(f)
        with cdna4.Session(d, max_seq=64) as s:
            outs.append(s.generate_ex(list(range(5, 30)), cdna4.GenerateCfg(9), with_logits=True))
    assert outs[0]["tokens"] == outs[1]["tokens"]
    assert np.isfinite(outs[0]["logits"]).all() and np.array_equal(outs[0]["logits"], outs[1]["logits"])
