"""GPU: bf16 rows counted by value (ws_code.h), through the C ABI against the CPU oracle on identical seeded inputs, at the sizes
where it can go wrong: vocabularies one token either side of a vector, of a round of the workgroup and of what the registers
hold, rows off every alignment, one and two copies of the counts, ties by the ten thousand with touched tokens among them, every
combination of filters, and the rows it hands back. Bars as in test_gpu_sample.py (gpu_cases.compare_rows)."""
import numpy as np
import pytest
import torch

import gpu_cases as gc

pytestmark = pytest.mark.gpu


def case(rows, V, n_hist=300, n_bias=20, allowed=None, seed=3, logits=None):
    c = gc.make_cfg2(rows=rows, V=V, n_hist=min(n_hist, V), n_bias=min(n_bias, V))
    rng = np.random.default_rng(seed)
    c["logits"], c["dtype"] = gc.f32_to_bf16_bits(c["logits"] if logits is None else logits), "bf16"
    c["top_p"] = np.minimum(c["top_p"], 0.99)
    if allowed is not None:
        words = (V + 31) // 32
        c["allow"] = np.ascontiguousarray(np.packbits(rng.random((rows, words * 32)) < allowed, axis=1, bitorder="little").view(np.uint32))
    return c


def run(c, hints=False, handed_back=0, max_differ=0, rng_mode=1):
    """One launch, every row against the oracle. hints False: a batch of which nothing is known; True: of the short-list kind where it
    is one. No workspace is asked for: the rows are one workgroup's."""
    m = gc.pkg()
    d = gc.upload(c, hints=hints, min_p_hint=hints)
    smp = gc.sampler_for(c, d, rng_mode, max_split=1).run()
    assert m.lib().ws_sample_batch_workspace_use(smp.desc) == m.WORK_NONE
    res = gc.compare_rows(c, smp, range(c["rows"]), rng_mode, check_kept=False)
    assert res["differ"] <= max_differ and res["exact"] + res["differ"] == c["rows"], res
    fl = smp.flags.cpu().numpy()
    assert int(((fl & m.FLAG_ROUTE_HANDED_BACK) != 0).sum()) == handed_back, fl
    kind = m.FLAG_ROUTE_SHORT if hints and (d["top_k_max"] or d["min_p_min"]) else (0 if d["top_k"] is not None else m.FLAG_ROUTE_LEAN)
    assert (fl[(fl & m.FLAG_ROUTE_HANDED_BACK) == 0] & m.FLAG_ROUTE_MASK == kind).all(), fl
    return smp


SIZES = [8, 9, 33, 1000, 8191, 8192, 8193, 40960, 40961, 81920, 81921, 122880, 122881, 151937, 155648, 155649, 163840, 163841, 200003, 262144]


@pytest.mark.parametrize("V", SIZES)
def test_vocabularies_off_every_boundary(V):
    run(case(3, V))


@pytest.mark.parametrize("V", [9, 8193, 50257, 163841])
@pytest.mark.parametrize("allowed", [0.1, 0.7])
def test_rows_with_an_allow_mask(V, allowed):
    c = case(4, V, allowed=allowed)
    c["allow"][:, 0] |= 7  # (no row without a token)
    run(c)


@pytest.mark.parametrize("V,n_hist,n_bias", [(50257, 1, 0), (50257, 0, 1), (50257, 0, 0), (50257, 2049, 2047), (151936, 4096, 300), (151936, 5000, 20), (151936, 2047, 0),
                                             (262144, 2500, 200), (20000, 7000, 0)])
def test_histories_and_bias_lists(V, n_hist, n_bias):
    """One and two ids a thread at hand and the ids behind them; tables that leave room for one copy of the counts."""
    c = case(3, V, n_hist=n_hist, n_bias=n_bias)
    if n_hist:
        c["hist"][0] = c["hist"][0] % 50  # (a text of few tokens)
        c["hist"][1, ::3] = [-1, V, 2 ** 31 - 1][n_hist % 3]  # (ids outside the vocabulary are nobody's)
    if n_bias > 10:
        c["bias_ids"][0, 5:10] = c["bias_ids"][0, 0]  # (several entries of one token, in listed order)
        c["bias_vals"][1, :4] = [40.0, 35.5, -300.0, 0.0]
    run(c)


@pytest.mark.parametrize("step,V,n_hist", [(0.5, 151937, 2000), (4.0, 60000, 300), (100.0, 30000, 100), (0.5, 200001, 500)])
def test_thousands_of_tied_tokens(step, V, n_hist):
    """Logits on a grid: every cut and draw falls among tokens that tie, thousands of them, which the lower ids win. With
    penalties that change nothing, touched tokens tie with the others; with small ones they lie just above and below."""
    rng = np.random.default_rng(5)
    x = (np.round(rng.standard_normal((6, V)) * 2 / step) * step).astype(np.float32) + 1.0
    c = case(6, V, n_hist=n_hist, n_bias=0, logits=x)
    c["rep"][:3] = 1.0
    c["pres"][:3] = c["freq"][:3] = 0.0
    c["pres"][3:] = [-1e-3, 1e-3, 0.0]
    c["top_k"][:] = [0, 0, 3000, 0, 500, 20]
    c["min_p"][:] = [0.0, 0.05, 0.0, 0.0, 0.0, 0.2]
    run(c)


@pytest.mark.parametrize("top_k,top_p,min_p", [(1, 0.9, 0.0), (1024, 1.0, 0.0), (40, 1.0, 0.1), (40, 0.5, 0.0), (0, 0.999, 0.0), (0, 1e-9, 0.0), (0, 1.0, 1.0), (0, 1.0, 1e-4), (0, 0.9, 0.01),
                                               (20000, 0.95, 0.0), (50000, 0.95, 0.0), (60000, 0.95, 0.0), (60000, 1.0, 0.0)])
@pytest.mark.parametrize("hints", [False, True])
def test_every_combination_of_filters(top_k, top_p, min_p, hints):
    """A top-k beyond the tokens a mask leaves, and beyond the vocabulary, among them."""
    c = case(4, 50001, allowed=0.6 if top_k >= 20000 else None)
    c["top_k"][:], c["top_p"][:], c["min_p"][:] = top_k, top_p, min_p
    run(c, hints=hints and top_k <= 1024, rng_mode=int(top_k) % 2, max_differ=1 if top_p == 0.999 else 0)  # (one cut lies within 1e-6 of a token's edge)


def test_short_list_batches_that_are_counted():
    """top-k 1000 in two parts' worth of rows, and a min-p without a top-k."""
    c = case(5, 60001)
    c["top_k"][:] = 1000
    run(c, hints=True)
    c["top_k"][:] = 0
    run(c, hints=True)


def test_rows_off_every_alignment_and_strides():
    m = gc.pkg()
    c = case(7, 40003, n_hist=0, n_bias=0)
    d = gc.upload(c)
    for stride in (40003, 40008, 41001):
        wide = torch.full((7, stride), float("inf"), dtype=torch.bfloat16, device="cuda:0")
        wide[:, :40003] = d["logits"]
        smp = gc.sampler_for(c, dict(d, logits=wide[:, :40003]), 1, max_split=1).run()
        res = gc.compare_rows(c, smp, range(7), 1, check_kept=False)
        assert res["exact"] == 7 and not ((smp.flags & m.FLAG_ROUTE_HANDED_BACK) != 0).any(), res


@pytest.mark.parametrize("hints", [False, True])
def test_a_token_far_above_the_head_of_the_row(hints):
    """The anchor of the masses comes from the row's first tokens; one far above it, and far below."""
    c = case(4, 50000, n_hist=30)
    x = gc.bf16_bits_to_f32(c["logits"]).copy()
    x[0, 40000] = 60.0
    x[1, 49999] = 300.0
    x[2, :20000] = 90.0
    c["allow"] = np.full((4, (50000 + 31) // 32), 0xffffffff, np.uint32)
    c["allow"][2, :20000 // 32] = 0  # (the head is masked out)
    x[3] -= 200.0
    c["logits"] = gc.f32_to_bf16_bits(x)
    if hints:
        c["top_k"][:] = 40
    run(c, hints=hints)


def test_rows_for_the_three_pass_code():
    """A logit of 512 and more, a NaN of either sign, logits that are all zero, a maximum near the last bin: answered by the three-pass code, the
    same. (A NaN with its sign set is in the tail already.)"""
    c = case(6, 20000, n_hist=50)
    x = gc.bf16_bits_to_f32(c["logits"]).copy()
    x[0, 100] = 512.0
    x[3] = 0.0
    x[4] -= 375.0
    c["logits"] = gc.f32_to_bf16_bits(x)
    c["logits"][1, 5] = 0x7fc0
    c["logits"][2, 5] = 0xffc0
    c["rep"][3] = 1.0
    c["pres"][3] = c["freq"][3] = 0.0
    c["bias_vals"][3] = 0.0
    c["rep"][4] = 1.0
    run(c, handed_back=4)


def test_the_same_cut_as_the_other_kernels():
    """Rows that keep some 17000 tokens, each six millionths of the mass: the single-sweep kernel (asked for a kept-set dump) cuts them at
    the same token, because the masses are the same."""
    for rows, max_split in ((24, 0), (24, 1)):
        c = gc.make_cfg3(rows=rows)
        c["top_k"][0] = 16000
        d = gc.upload(c)
        a = gc.sampler_for(c, d, 1, max_split=max_split).run()
        b = gc.sampler_for(c, d, 1, kept_cap=8, max_split=max_split).run()
        torch.cuda.synchronize()
        assert int((a.n_kept != b.n_kept).sum()) <= 1 and int((a.token != b.token).sum()) <= 1
        assert torch.equal(a.stats[:, 0], b.stats[:, 0]) and torch.allclose(a.stats[:, 1], b.stats[:, 1], rtol=2e-7, atol=0)


def test_captured_and_replayed():
    """Nothing but one kernel: a captured launch, replayed with eager work in between."""
    c = case(5, 50257)
    smp = gc.sampler_for(c, gc.upload(c), 1)
    smp.run()
    torch.cuda.synchronize()
    want = [t.clone() for t in (smp.token, smp.prob, smp.n_kept, smp.stats)]
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        smp.run()
        s.synchronize()
        with torch.cuda.graph(g, stream=s):
            smp.run()
    for _ in range(3):
        for t in (smp.token, smp.prob, smp.n_kept, smp.stats):
            t.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(want, (smp.token, smp.prob, smp.n_kept, smp.stats)))


@pytest.mark.parametrize("V,allowed,n_hist", [(9, None, 0), (255, None, 20), (257, None, 20), (8193, None, 300), (50257, 0.5, 300), (151936, None, 2000), (163841, None, 100), (262144, 0.9, 0)])
def test_rows_without_a_filter(V, allowed, n_hist):
    """Their short list is the 256 largest; a draw behind it walks the others in id order. Flat and peaked rows, tokens tied with the
    256th, and touched tokens on either side of it."""
    m = gc.pkg()
    c = case(16, V, n_hist=n_hist, n_bias=5, allowed=allowed)
    x = gc.bf16_bits_to_f32(c["logits"]).copy()
    x[:4] *= 3.0
    x[8:12] = np.round(x[8:12]) + 0.5
    c["logits"] = gc.f32_to_bf16_bits(x)
    if allowed is not None:
        c["allow"][:, 0] |= 7
    c["top_k"][:], c["top_p"][:], c["min_p"][:] = 0, 1.0, 0.0
    smp = run(c, max_differ=1)
    assert ((smp.flags & 64) != 0).all()  # (WS_FLAG_OPEN)


# A row's largest tokens by their octave: at the low and at the high end of a group of eight values, and between.
PEAKS = [9.0, 9.4375, 10.02, 16.0, 16.875, 17.05, 20.45, 24.05, 33.3, 38.0, 70.2, 301.0]
TEMPERATURES = [2e-4, 2.5e-4, 1e-3, 0.01, 0.02, 0.03, 0.05, 0.1, 0.3]


def cold_case(T, kind, hints, V=50001):
    """Rows whose largest tokens lie a few e-folds apart at temperature T. kind "bias" and "history": tokens at any float, by a bias or by
    penalties, untouched ones at the next values below them; "plain": no touched token at all; "beside": a touched token far below, the others on the grid."""
    n = len(PEAKS)
    c = case(2 * n, V, n_hist=0 if kind == "plain" else 40, n_bias=0 if kind == "plain" else 12)
    rng = np.random.default_rng(int(T * 1000) + len(kind))
    x = gc.bf16_bits_to_f32(c["logits"]).copy()
    c["inv_t"][:] = np.float32(1.0) / np.float32(T)
    c["rep"][:], c["pres"][:], c["freq"][:] = 1.1, 0.3, 0.02
    for r in range(2 * n):
        peak, at = np.float32(PEAKS[r // 2]), rng.permutation(V)
        step = np.float32(2.0 ** (np.floor(np.log2(peak)) - 7))
        low = np.float32(np.floor(peak / step) * step)  # the largest value at or below the peak
        if kind in ("plain", "beside"):
            x[r, at[:6]] = low - step * np.array([0, 0, 1, 1, 2, 5], np.float32)
        else:
            x[r, at[20:26]] = low - step * np.array([1, 1, 2, 3, 4, 9], np.float32)
        if kind == "plain":
            continue
        c["bias_ids"][r], c["bias_vals"][r] = at[:12] if kind == "bias" else at[30:42], rng.uniform(-3, 0, 12)
        c["hist"][r, :8] = at[50:58] if kind == "bias" else at[:8]
        c["hist"][r, 8:] = at[60:92]
        if kind == "bias":
            c["bias_vals"][r] = peak - T * np.array([0, 0.2, 0.5, 0.9, 1.3, 2.1, 3.0, 4.2, 6.0, 9.0, 14.0, 20.0]) - x[r, at[:12]]
        elif kind == "history":  # (raw values whose penalised ones lie around the peak)
            x[r, at[:8]] = np.float32((peak + 0.32) * 1.1) - step * np.arange(8, dtype=np.float32)
    c["logits"] = gc.f32_to_bf16_bits(x)
    filters = [(0, 0.9, 0.0), (40, 1.0, 0.0), (0, 0.95, 0.05), (40, 0.7, 0.0), (0, 1.0, 0.02), (3, 1.0, 0.0), (1000, 0.99, 0.0), (0, 1.0, 0.0)]
    if hints:
        filters = [f for f in filters if f[0] or f[2]]
    for r in range(2 * n):
        c["top_k"][r], c["top_p"][r], c["min_p"][r] = filters[(r * 5 + r // len(filters)) % len(filters)]
    return c


@pytest.mark.parametrize("hints", [False, True])
@pytest.mark.parametrize("T", TEMPERATURES)
@pytest.mark.parametrize("kind", ["bias", "history", "beside", "plain"])
def test_cold_rows(kind, T, hints):
    """Octaves are many e-folds wide at low temperatures, and so are the groups of eight values that masses are added up in: hundreds of e-folds, more
    than 64 bits have room for. Below a temperature of 1/4096 the rows are the three-pass code's."""
    c = cold_case(T, kind, hints)
    run(c, hints=hints, handed_back=c["rows"] if T < 1 / 4096 else 0)


@pytest.mark.parametrize("allowed", [None, 0.5])
@pytest.mark.parametrize("hints", [False, True])
def test_hot_rows_and_floors_below_the_last_bin(hints, allowed):
    """Temperatures at which the last bin is not 50 e-folds below the maximum, and min-p floors that lie below it: nothing is left out
    as long as every token that is not masked out has a bin of its own."""
    c = case(12, 50001, allowed=allowed)
    c["inv_t"][:] = 1 / np.array([8.0, 10.0, 30.0, 1.0, 1.0, 0.7] * 2)
    c["min_p"][:] = [0.05, 0.0, 0.3, 1e-200, 1e-300, 1e-250] * 2
    c["top_k"][:] = [0, 50, 0, 0, 60000, 45000] * 2
    c["top_p"][:] = [1.0, 0.9, 1.0, 1.0, 1.0, 1.0, 0.9, 1.0, 0.99, 0.9, 0.9, 1.0]
    if hints:
        c["top_k"][:] = [0, 50, 0, 0, 1000, 500] * 2
        c["min_p"][3::6] = 1e-3
    run(c, hints=hints)
    x = gc.bf16_bits_to_f32(c["logits"]).copy()
    x[:, 17] = -400.0  # (a token in the last bins: the rows are the three-pass code's, but for the one whose floor lies above it)
    c["logits"] = gc.f32_to_bf16_bits(x)
    if allowed is not None:
        c["allow"][:, 0] |= 1 << 17
    run(c, hints=hints, handed_back=10 if hints else 12)


@pytest.mark.parametrize("n_hist,n_bias", [(29, 0), (30, 2), (0, 29)])
def test_more_entries_than_the_batch_declares(n_hist, n_bias):
    """The tables are rounded up to four entries: a row that has one to three more than max_hist and max_bias say is refused all the same."""
    m = gc.pkg()
    c = case(5, 50001, n_hist=n_hist, n_bias=n_bias)
    smp = gc.sampler_for(c, gc.upload(c), 1, max_split=1)
    if n_hist:
        smp.desc.max_hist -= 1
    else:
        smp.desc.max_bias -= 1
    smp.run()
    assert ((smp.flags & m.FLAG_BAD_PARAM) != 0).all() and (smp.token == -1).all(), smp.flags
