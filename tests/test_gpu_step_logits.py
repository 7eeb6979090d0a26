"""Logits of every step through the session's pinned slots: calls of fewer, as many and more steps than
slots, in any order on one session, give the rows of one long call; without logits the same tokens."""
import numpy as np
import pytest

import cdna4
from cdna4 import model_format

pytestmark = pytest.mark.gpu


def test_rows_do_not_depend_on_the_number_of_steps(tmp_path):
    model_format.random_model(str(tmp_path), n_layers=2, hidden=128, n_heads=2, ffn_dim=256, vocab_size=1003, seed=4)
    ids = list(range(7, 40))
    with cdna4.Session(str(tmp_path), max_seq=96) as s:
        want = s.generate_ex(ids, cdna4.GenerateCfg(23), with_logits=True)
        assert np.isfinite(want["logits"]).all()
        for new in (1, 5, 4, 3, 9, 1, 8, 23):
            got = s.generate_ex(ids, cdna4.GenerateCfg(new), with_logits=True)
            assert got["tokens"] == want["tokens"][:new], new
            assert np.array_equal(got["logits"], want["logits"][:new]), new
        stop = want["tokens"][6]   # ends by the token: fewer rows than asked for
        got = s.generate_ex(ids, cdna4.GenerateCfg(23, stop), with_logits=True)
        n = len(got["tokens"])
        assert got["tokens"] == want["tokens"][:n] and np.array_equal(got["logits"], want["logits"][:n])
        assert s.generate_ex(ids, cdna4.GenerateCfg(23))["tokens"] == want["tokens"]
