"""GPU: tokens that a bias list names several times, through every sampler kernel, against the CPU oracle: entries next to each other and
hundreds apart, first and last of the list, many such tokens in one wave, tokens of the history among them. The largest logit of a row is such a
token's, so that the row's maximum - compared to the bit - says in which order its entries were added. Bars as in test_gpu_sample.py."""
import numpy as np
import pytest

import gpu_cases as gc

pytestmark = pytest.mark.gpu

KINDS = {  # name: (rows, V, dtype, hints, top_k, max_split)
    "few": (3, 50257, "f32", True, 40, 0),
    "short": (3, 50257, "f32", True, 40, 1),
    "twin": (300, 8209, "f32", True, 40, 0),
    "lean": (3, 50264, "f32", True, 0, 1),
    "single sweep": (3, 50264, "f32", False, 40, 1),
    "split": (3, 70000, "f32", False, 40, 4),
    "three-pass": (3, 50257, "f32", False, 40, 1),
    "bf16": (3, 50257, "bf16", False, 40, 1),
    "bf16 short": (300, 8209, "bf16", True, 40, 0),
}


@pytest.mark.parametrize("n_bias", [2, 64, 65, 300, 1500])
@pytest.mark.parametrize("kind", list(KINDS))
def test_tokens_with_several_bias_entries(kind, n_bias):
    rows, V, dtype, hints, top_k, max_split = KINDS[kind]
    c = gc.make_cfg2(rows=rows, V=V, n_hist=600, n_bias=n_bias)
    rng = np.random.default_rng(n_bias)
    c["top_k"][:] = top_k
    c["top_p"][:] = 0.9
    if not top_k:
        c["min_p"][:] = 0.0
    x = c["logits"]
    for r in range(rows):
        at = rng.permutation(n_bias)
        at = np.concatenate([[0, n_bias - 1], at[(at != 0) & (at != n_bias - 1)]])  # (the first and the last entry are one token's)
        token, k = rng.permutation(V), 0
        while len(at) >= 2 and k < 60:
            n = min(len(at), int(rng.integers(2, 8)))
            c["bias_ids"][r, at[:n]] = token[k] if k % 3 else c["hist"][r, k]
            if k == 0:
                x[r, c["hist"][r, 0]] = 30.0
            at, k = at[n:], k + 1
    c["bias_vals"] = (c["bias_vals"] * 0.31).astype(np.float32)
    if dtype == "bf16":
        c["logits"], c["dtype"] = gc.f32_to_bf16_bits(x), "bf16"
    d = gc.upload(c, hints=hints)
    if kind == "lean":
        assert d["top_k"] is None
        d["min_p_min"] = 0.0
    smp = gc.sampler_for(c, d, 1, max_split=max_split).run()
    which = range(rows) if rows < 10 else range(0, rows, 23)
    res = gc.compare_rows(c, smp, which, 1, check_kept=False)
    assert res["exact"] + res["differ"] == res["rows"] and res["differ"] == 0, res
