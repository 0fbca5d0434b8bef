"""GPU: the one-sweep kernel for batches without a top-k (fp32 and bf16 rows, ws_batch.top_k = NULL, no kept-set dump)
through the C ABI against the CPU oracle on identical seeded inputs.

Bars as in test_gpu_sample.py: token, kept count, row maximum identical, the token's probability and the normaliser
within 1e-6 relative; a row may differ from the oracle only where the device reports WS_FLAG_NEAR_*, and every test
states how many such rows it allows. Every test also states which way the rows went (WS_FLAG_ROUTE_*): a test of this
kernel that silently ran another one proves nothing."""
import numpy as np
import pytest
import torch

import gpu_cases as gc

pytestmark = pytest.mark.gpu


def _no_top_k(c):
    c["top_k"][:] = 0
    return c


def run_lean(c, rng_mode, rows=None, max_differ=0, handed_back=0, **more):
    """One launch without a kept-set dump; the rows against the oracle; the route census."""
    m = gc.pkg()
    assert not c["top_k"].any()
    d = gc.upload(c, hints=True)
    assert d["top_k"] is None
    d["min_p_min"] = 0.0  # (a batch that says its rows have a min-p goes to the short-list kernel: not this test's)
    smp = gc.sampler_for(c, d, rng_mode, max_split=1, **more).run()
    rows = range(c["rows"]) if rows is None else rows
    res = gc.compare_rows(c, smp, rows, rng_mode, check_kept=False)
    assert res["differ"] <= max_differ and res["exact"] + res["differ"] == res["rows"], res
    fl = smp.flags.cpu().numpy()
    lean = int(((fl & m.FLAG_ROUTE_LEAN) != 0).sum())
    back = int(((fl & m.FLAG_ROUTE_HANDED_BACK) != 0).sum())
    assert lean + back == c["rows"] and back <= handed_back, (lean, back, c["rows"])
    res.update(lean=lean, handed_back=back)
    return res, smp


def test_north_star_tile_every_row():
    """256 x 151936, penalties over 2048-id histories, top-p 0.9: every row through the one-sweep kernel, every row
    against the oracle."""
    c = gc.make_tile()
    res, _ = run_lean(c, 1)
    assert res["exact"] == 256 and res["lean"] == 256, res
    print(res)


@pytest.mark.parametrize("rng_mode", [0, 1])
def test_min_p_top_p_bias_and_long_histories(rng_mode):
    """cfg2's rows without their top-k: temperatures 0.5 .. 1.2, top-p 0.8 .. 1, min-p 0.05, 300 bias entries, 4096-id
    histories (four ids a thread in the collect)."""
    c = _no_top_k(gc.make_cfg2(rows=24))
    res, _ = run_lean(c, rng_mode)
    assert res["exact"] == 24 and res["lean"] == 24, res
    print(res)


def test_min_p_only_and_top_p_only_rows_and_short_histories():
    c = _no_top_k(gc.make_cfg2(rows=16, V=151936, n_hist=300, n_bias=0))
    c["top_p"][:8] = 1.0
    c["min_p"][:8] = [0.5, 0.2, 0.05, 0.01, 0.001, 1e-4, 0.9, 1.0]
    c["min_p"][8:] = 0.0
    c["top_p"][8:] = [0.1, 0.5, 0.9, 0.95, 0.99, 0.999, 0.9999, 0.3]
    res, _ = run_lean(c, 1, max_differ=1, handed_back=2)  # (top-p 0.9999: the cut falls in a bin of more tokens than the finish takes)
    assert res["exact"] >= 15 and res["lean"] >= 14, res
    print(res)


def test_rows_with_an_allow_mask():
    """90 % of the tokens masked out, bias entries on masked and unmasked tokens alike."""
    c = _no_top_k(gc.make_cfg5(rows=12, V=151936, n_hist=2048, n_bias=200))
    res, _ = run_lean(c, 1, handed_back=1)
    assert res["exact"] == 12 and res["lean"] >= 11, res
    print(res)


@pytest.mark.parametrize("V", [8200, 65536, 100000, 163840])
def test_other_vocabularies(V):
    """Rows that end in the middle of a round of the 1024 threads, that fill a few registers of the bin cache only, and
    the longest the cache holds."""
    c = _no_top_k(gc.make_cfg2(rows=8, V=V, n_hist=min(V // 4, 1000), n_bias=50))
    res, _ = run_lean(c, 1, handed_back=1)  # (one row's top-p is 0.998: its cut bin holds more tokens than the finish takes)
    assert res["exact"] == 8 and res["lean"] >= 7, res
    print(res)


@pytest.mark.parametrize("V,masked,lists", [(V, masked, lists) for V in (8193, 8195, 16386, 20481, 32771, 50257, 71348, 102397, 102398, 102399, 151937, 163837, 163839)
                                            for masked in (False, True) for lists in (False, True)
                                            if lists or V >= (32768 if masked else 20480)])  # (shorter rows without lists are swept three times)
def test_rows_off_every_boundary(V, masked, lists):
    """Rows of any length, which begin at any address: those that end inside a vector, one token either side of a round; with touched tokens, the largest
    logits and masked-out tokens in the last vector, and mask bits set behind the row's end."""
    c = _no_top_k(gc.make_cfg2(rows=6, V=V, n_hist=700 if lists else 0, n_bias=50 if lists else 0))
    c["top_p"] = np.minimum(c["top_p"], 0.95)
    rng = np.random.default_rng(V)
    for r in range(6):
        if lists:
            c["hist"][r][:2] = [V - 1, V - 1 - r % 4]
        c["logits"][r, V - 1 - (r * 3) % 8] = 9.0 + r
    if masked:
        c["allow"] = rng.integers(0, 1 << 32, (6, (V + 31) // 32), dtype=np.uint64).astype(np.uint32) | np.uint32(0x10000001)
        c["logits"][:2, :500:40] = 14.0  # (some of them masked out: far above the others)
    res, _ = run_lean(c, 1, handed_back=2 if masked else 1)
    assert res["exact"] == 6, res


def test_no_history_no_bias_no_penalties():
    c = _no_top_k(gc.make_cfg2(rows=8, V=151936, n_hist=0, n_bias=0))
    res, _ = run_lean(c, 0, handed_back=1)
    assert res["exact"] == 8 and res["lean"] >= 7, res


def test_thousands_of_equal_logits_at_the_cut():
    """Logits rounded to one decimal: every cut falls among thousands of ties, which the lower ids win
    (src/sampling/sampler.cpp:18-21). Up to 4096 candidates a row are sorted in place; a row with more goes to the
    three-pass code inside the launch and says so. Either way the answers are the oracle's."""
    c = _no_top_k(gc.make_cfg2(rows=8, V=151936, n_hist=500, n_bias=20))
    c["logits"] = np.round(c["logits"], 1)
    res, smp = run_lean(c, 1, max_differ=1, handed_back=8)
    assert res["exact"] >= 7 and res["lean"] >= 1, res
    print(res)


def _as_bf16(c):
    c["logits"] = gc.f32_to_bf16_bits(c["logits"])
    c["dtype"] = "bf16"
    return c


def test_bf16_zipfian_rows_with_hundreds_of_ties_at_the_cut():
    """cfg3's rows: bf16, -1.1 ln(rank) + noise, top-p 0.9 - some 17000 tokens kept, and the cut among the several
    hundred that share its bf16 value."""
    c = gc.make_cfg3(rows=64)
    # (two of these rows have their cut within 1e-7 of a token's edge and are reported as such, by every kernel here)
    res, _ = run_lean(c, 1, max_differ=2, handed_back=2)
    assert res["exact"] >= 62 and res["lean"] >= 62, res
    print(res)


def test_bf16_ties_from_hundreds_to_thousands_at_the_cut():
    """The same rows with top-p from 0.8 to 0.985: the deeper the cut, the more tokens share its bf16 value - 500 to
    beyond the 4096 a row that the kernel sorts in place (one, two, three and four candidates a thread, the 1024
    buckets and the 256); the rows beyond are handed back. Every answer is the oracle's either way."""
    c = gc.make_cfg3(rows=18)
    c["top_p"][:] = np.repeat([0.8, 0.9, 0.93, 0.95, 0.97, 0.985], 3)
    res, _ = run_lean(c, 0, max_differ=2, handed_back=9)
    assert res["exact"] >= 16 and res["lean"] >= 9, res
    print(res)


@pytest.mark.parametrize("rng_mode", [0, 1])
def test_bf16_min_p_top_p_bias_and_long_histories(rng_mode):
    c = _as_bf16(_no_top_k(gc.make_cfg2(rows=24)))
    res, _ = run_lean(c, rng_mode, max_differ=1, handed_back=1)
    assert res["exact"] >= 23 and res["lean"] >= 23, res
    print(res)


def test_bf16_rows_with_an_allow_mask():
    c = _as_bf16(_no_top_k(gc.make_cfg5(rows=12, V=151936, n_hist=2048, n_bias=200)))
    res, _ = run_lean(c, 1, max_differ=1, handed_back=1)
    assert res["exact"] >= 11 and res["lean"] >= 11, res
    print(res)


@pytest.mark.parametrize("V", [8200, 65536, 100000, 163840])
def test_bf16_other_vocabularies(V):
    c = _as_bf16(_no_top_k(gc.make_cfg2(rows=8, V=V, n_hist=min(V // 4, 1000), n_bias=50)))
    res, _ = run_lean(c, 1, max_differ=1, handed_back=1)
    assert res["exact"] >= 7 and res["lean"] >= 7, res
    print(res)


def test_outlier_above_the_head_of_the_row_is_handed_back():
    """The anchor comes from the first 8192 tokens; a token far above it later in the row breaks the bound."""
    c = _no_top_k(gc.make_cfg2(rows=4, V=151936, n_hist=300, n_bias=0))
    c["logits"][1, 100000] = 60.0
    c["logits"][3, 151935] = 35.0
    res, _ = run_lean(c, 1, handed_back=2)
    assert res["exact"] == 4 and res["handed_back"] == 2, res


def test_same_answers_as_the_kernel_that_takes_a_top_k():
    """The same batch with top_k given as an array of zeros goes through the other single-sweep kernel: same tokens, kept
    counts and maxima, probabilities within 1e-6 (on the rows that neither reports near a boundary)."""
    m = gc.pkg()
    c = _no_top_k(gc.make_tile(rows=160))
    d = gc.upload(c, hints=True)
    a = gc.sampler_for(c, d, 1, max_split=1).run()
    d["top_k"] = torch.zeros(c["rows"], dtype=torch.int32, device="cuda:0")
    b = gc.sampler_for(c, d, 1, max_split=1).run()
    torch.cuda.synchronize()
    assert ((a.flags & m.FLAG_ROUTE_LEAN) != 0).all() and ((b.flags & m.FLAG_ROUTE_LEAN) == 0).all()
    # (The two kernels count their bins from different anchors, so their sums round differently in the last place: a
    # row that either of them reports within tolerance of a boundary may come out on either side. Everywhere else the
    # answers are the same.)
    sure = ((a.flags | b.flags) & m.FLAG_NEAR) == 0
    assert int(sure.sum()) >= c["rows"] // 2
    for name in ("token", "n_kept"):
        assert torch.equal(getattr(a, name)[sure], getattr(b, name)[sure]), name
    differ = int((a.n_kept != b.n_kept).sum() + (a.token != b.token).sum())
    assert differ <= 2, differ
    assert torch.equal(a.stats[:, 0], b.stats[:, 0])
    assert torch.allclose(a.prob[sure], b.prob[sure], rtol=1e-6, atol=0)


def _ragged(kind, sigma, V, rows, seed):
    """Rows of V tokens on the GPU: N(0, sigma), a few tokens raised to 10 .. 14, or Zipfian."""
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    x = torch.empty((rows, V), device="cuda:0").normal_(0.0, sigma, generator=g)
    if kind == "raised":
        ids = torch.randint(0, V, (rows, 20), device="cuda:0", generator=g)
        x.scatter_(1, ids, torch.empty((rows, 20), device="cuda:0").uniform_(10.0, 14.0, generator=g))
    elif kind == "zipf":
        base = -1.1 * torch.log(torch.arange(1, V + 1, device="cuda:0", dtype=torch.float32))
        x += base[torch.rand((rows, V), device="cuda:0", generator=g).argsort(dim=1)]
    return x, torch.empty(rows, device="cuda:0").uniform_(0.7, 1.7, generator=g)


def _sampled(x, inv_t, **more):
    m, rows = gc.pkg(), x.shape[0]
    steps = torch.arange(rows, dtype=torch.int64, device="cuda:0")
    return m.BatchSampler(x, inv_t, steps * 77 + 5, steps, top_p=torch.full((rows,), 0.9, dtype=torch.float64, device="cuda:0"), rng=1, max_split=1, **more).run()


@pytest.mark.parametrize("kind,sigma,V", [("normal", 3.0, 50257), ("normal", 1.5, 20483), ("raised", 2.0, 151937), ("raised", 3.0, 99991), ("zipf", 0.4, 151937)])
def test_normaliser_as_close_as_three_sweeps(kind, sigma, V):
    """Rows off every boundary, whose masses come from the bins: no further from 64 bits than where the same rows are swept three times (a kept-set dump takes
    them there), and the same number on nearly every row - both count from eight units above the row's head, and only the order of the 64-bit sums is another.
    The rows whose maximum lies above that (the three sweeps take it for the anchor then) are looked at by themselves: a coordinate of up to 256 is off by
    2^-17, a mass by 2^-17 / 64 = 1.2e-7 at most, and the result's own rounding is 6e-8."""
    m = gc.pkg()
    x, inv_t = _ragged(kind, sigma, V, 128, V)
    a, b = _sampled(x, inv_t), _sampled(x, inv_t, kept_cap=8)
    torch.cuda.synchronize()
    lean = (a.flags & m.FLAG_ROUTE_MASK) == m.FLAG_ROUTE_LEAN
    assert int(lean.sum()) >= 120 and ((b.flags & m.FLAG_ROUTE_LEAN) == 0).all()
    top = x.double().amax(1, keepdim=True)
    z = torch.exp((x.double() - top) * inv_t.double()[:, None]).sum(1)
    off = [s.stats[:, 1].double() / z - 1.0 for s in (a, b)]
    lies = (top[:, 0] - x[:, :8192].double().amax(1)) * inv_t.double()
    below, over = lean & (lies < 7.9), lean & (lies >= 7.9)
    assert int(below.sum()) >= 64
    rms = [float(o[below].square().mean().sqrt()) for o in off]
    assert rms[0] <= 1.05 * rms[1] + 2e-9, rms
    assert float((a.stats[below, 1] == b.stats[below, 1]).double().mean()) >= 0.95
    if over.any():
        assert float(off[0][over].abs().max()) <= 1.2e-7 + 6e-8
    same = below & (((a.flags | b.flags) & m.FLAG_NEAR) == 0)
    assert int(same.sum()) >= 32 and torch.equal(a.n_kept[same], b.n_kept[same]) and torch.equal(a.token[same], b.token[same])
    print(kind, V, rms)


@pytest.mark.parametrize("V", [50257, 151936, 151937])
@pytest.mark.parametrize("lists,masked", [(False, False), (True, False), (True, True)])
def test_maximum_above_the_bins_is_swept_once_more(V, lists, masked):
    """Rows whose maximum lies 11 to 31 units of the exponent above the largest of their first 8192 tokens - a token late in the row, alone or with others just
    below it - are read a second time by the same code when it is more than 12, and not handed back. Their masses are as good as any: the
    second sweep counts from the maximum."""
    m = gc.pkg()
    units = [11.0, 13.0, 16.0, 20.0, 25.0, 31.0]
    c = _no_top_k(gc.make_cfg2(rows=6, V=V, n_hist=400 if lists else 0, n_bias=40 if lists else 0))
    c["top_p"] = np.minimum(c["top_p"], 0.95)
    c["min_p"][:] = 0.0
    if masked:
        rng = np.random.default_rng(V)
        c["allow"] = rng.integers(0, 1 << 32, (6, (V + 31) // 32), dtype=np.uint64).astype(np.uint32)
    for r in range(6):
        late = V - 5 - 40 * r
        allowed = np.unpackbits(c["allow"][r].view(np.uint8), bitorder="little")[:8192].astype(bool) if masked else np.ones(8192, bool)
        head = float(c["logits"][r, :8192][allowed].max())
        for j in range(6 if r % 2 else 1):
            at = late - 7 * j
            c["logits"][r, at] = head + (units[r] - 0.4 * j) / float(c["inv_t"][r])
            if masked:
                c["allow"][r, at >> 5] |= np.uint32(1 << (at & 31))
            if lists:  # (nothing moves these tokens)
                c["hist"][r][c["hist"][r] == at] = 0
                c["bias_ids"][r][c["bias_ids"][r] == at] = 0
    res, smp = run_lean(c, 1)
    fl = smp.flags.cpu().numpy()
    assert res["exact"] == 6 and res["handed_back"] == 0, res
    again = (fl & m.FLAG_ROUTE_REDONE) != 0
    assert not again[0] and again[1:].all(), fl
    x = torch.from_numpy(c["logits"]).double()
    if not lists:
        z = torch.exp((x - x.amax(1, keepdim=True)) * torch.from_numpy(c["inv_t"]).double()[:, None]).sum(1).numpy()
        off = smp.stats[:, 1].cpu().numpy().astype(np.float64) / z - 1.0
        assert np.abs(off[again]).max() <= 2.4e-7, off  # (coordinates below 512: 2^-16 / 64 at most, and the result's rounding is 6e-8)


@pytest.mark.parametrize("V", [50256, 50257, 151937])
@pytest.mark.parametrize("lists", [False, True])
def test_rows_without_any_filter(V, lists):
    """A batch that has neither a top-p nor a min-p is nothing for this kernel, which would hand back every row. Rows off the vector boundaries go straight to
    the three sweeps, with the workspace that takes their touched tokens' logits; the others to the single-sweep kernel."""
    m = gc.pkg()
    c = _no_top_k(gc.make_cfg2(rows=5, V=V, n_hist=600 if lists else 0, n_bias=30 if lists else 0))
    c["top_p"][:], c["min_p"][:] = 1.0, 0.0
    d = gc.upload(c, hints=True)
    d["top_p"] = d["min_p"] = None
    d["min_p_min"] = 0.0
    smp = gc.sampler_for(c, d, 1, max_split=1).run()
    res = gc.compare_rows(c, smp, range(5), 1, check_kept=False)
    assert res["exact"] + res["differ"] == 5 and res["differ"] <= 1, res
    assert not (smp.flags & (m.FLAG_ROUTE_LEAN | m.FLAG_ROUTE_HANDED_BACK)).any(), smp.flags
    use = m.lib().ws_sample_batch_workspace_use(smp.desc)
    tables = lists and V % 8 != 0
    assert use == (m.WORK_TABLES if tables else m.WORK_NONE) and (not tables or smp.workspace.numel() >= 5 * 8 * 630)


@pytest.mark.parametrize("V,ids,masked,lean", [
    (8191, 128, False, False), (8193, 127, False, False), (8193, 128, False, True), (16383, 127, False, False), (16385, 1, False, True), (20477, 0, False, False),
    (20481, 0, False, True), (8193, 511, True, False), (8193, 512, True, True), (20479, 511, True, False), (20481, 1, True, True), (32767, 0, True, False), (32769, 0, True, True)])
def test_short_rows_off_the_boundaries(V, ids, masked, lean):
    """Either side of the lengths from which rows that are not whole aligned vectors go this way: with no lists, with a few ids, with more; masked and not."""
    m = gc.pkg()
    c = _no_top_k(gc.make_cfg2(rows=3, V=V, n_hist=ids, n_bias=0))
    c["top_p"], c["min_p"][:] = np.minimum(c["top_p"], 0.95), 0.0
    if masked:
        c["allow"] = np.random.default_rng(V).integers(0, 1 << 32, (3, (V + 31) // 32), dtype=np.uint64).astype(np.uint32)
    d = gc.upload(c, hints=True)
    d["min_p_min"] = 0.0
    smp = gc.sampler_for(c, d, 1, max_split=1).run()
    res = gc.compare_rows(c, smp, range(3), 1, check_kept=False)
    assert res["exact"] == 3, res
    assert (((smp.flags & m.FLAG_ROUTE_LEAN) != 0) == lean).all(), smp.flags


@pytest.mark.parametrize("V,masked,n_hist", [(V, masked, n_hist) for V in (163841, 163844, 163848, 172032, 200003, 262136, 262143, 262144) for masked in (False, True) for n_hist in (0, 700)] +
                         [(262144, True, 3000), (200000, False, 4000)])
def test_rows_longer_than_the_shorter_bin_cache(V, masked, n_hist):
    """Rows of 163841 to 262144 tokens, one sweep as well: whole vectors and not, whole rounds and not, with touched tokens, the largest logits and masked-out
    tokens in the last vector."""
    c = _no_top_k(gc.make_cfg2(rows=5, V=V, n_hist=n_hist, n_bias=50 if n_hist else 0))
    c["top_p"] = np.minimum(c["top_p"], 0.95)
    for r in range(5):
        if n_hist:
            c["hist"][r][:2] = [V - 1, V - 1 - r % 4]
        c["logits"][r, V - 1 - (r * 3) % 8] = 9.0 + r
    if masked:
        rng = np.random.default_rng(V)
        c["allow"] = rng.integers(0, 1 << 32, (5, (V + 31) // 32), dtype=np.uint64).astype(np.uint32) | np.uint32(0x10000001)
        c["logits"][:2, :500:40] = 14.0
    res, _ = run_lean(c, 1, handed_back=1)
    assert res["exact"] == 5, res


@pytest.mark.parametrize("lists,masked", [(False, False), (True, True)])
def test_long_rows_are_swept_once_more_as_well(lists, masked):
    test_maximum_above_the_bins_is_swept_once_more(262144, lists, masked)


@pytest.mark.parametrize("kind,sigma,V", [("normal", 2.0, 262144), ("zipf", 0.4, 200003)])
def test_normaliser_of_long_rows(kind, sigma, V):
    test_normaliser_as_close_as_three_sweeps(kind, sigma, V)


@pytest.mark.parametrize("V,masked", [(262144, False), (200003, True)])
def test_more_finds_than_the_list_holds(V, masked):
    """The cut and the draw fall among 3000 tokens, and 20000 others lie 256 bins below those: their cached bytes are the same, and all are found. A long row
    looks at each before it lists it; it is not handed back."""
    c = _no_top_k(gc.make_cfg2(rows=4, V=V, n_hist=64, n_bias=8))
    c["inv_t"][:], c["top_p"][:], c["min_p"][:] = 1.0, 0.8, 0.0
    rng = np.random.default_rng(V)
    for r in range(4):
        x = np.full(V, -30.0, np.float32)
        at = rng.permutation(V)[:23000]
        x[at] = -1.0 + rng.uniform(0.0, 0.012, 23000).astype(np.float32)
        x[at[3000:]] -= 4.0
        c["logits"][r] = x
    if masked:
        c["allow"] = (rng.random((4, (V + 31) // 32 * 32)) < 0.9)
        c["allow"] = np.ascontiguousarray(np.packbits(c["allow"], axis=1, bitorder="little").view(np.uint32))
    res, _ = run_lean(c, 1)
    assert res["exact"] == 4 and res["handed_back"] == 0, res


@pytest.mark.parametrize("V,share", [(50257, 0.02), (151936, 0.17), (262144, 0.5)])
def test_masked_out_tokens_under_every_byte(V, share):
    """Nearly all of a row masked out, and cuts and draws under many different bytes (temperatures from 0.3 to 2): what is masked out is found with every one
    of them and dropped."""
    c = _no_top_k(gc.make_cfg2(rows=16, V=V, n_hist=100, n_bias=20))
    c["top_p"] = np.linspace(0.5, 0.95, 16)
    c["inv_t"] = np.linspace(0.5, 3.3, 16).astype(np.float32)
    c["min_p"][:] = 0.0
    rng = np.random.default_rng(V)
    c["allow"] = np.ascontiguousarray(np.packbits(rng.random((16, (V + 31) // 32 * 32)) < share, axis=1, bitorder="little").view(np.uint32))
    res, _ = run_lean(c, 1, max_differ=1, handed_back=1)
    assert res["exact"] >= 15, res


@pytest.mark.parametrize("V", [V + d for V in (32768, 49152, 65536, 98304, 131072, 155648, 163840) for d in (0, 1, 8)])
@pytest.mark.parametrize("masked", [False, True])
def test_rows_at_the_ends_of_the_bin_caches(V, masked):
    """One token more than a build's bin cache holds, and a row that fills it: the largest logits and touched tokens in the last vector."""
    c = _no_top_k(gc.make_cfg2(rows=3, V=V, n_hist=600, n_bias=30))
    c["top_p"] = np.minimum(c["top_p"], 0.95)
    for r in range(3):
        c["hist"][r][:2] = [V - 1, V - 1 - r]
        c["logits"][r, V - 1 - (r * 3) % 8] = 9.0 + r
    if masked:
        rng = np.random.default_rng(V)
        c["allow"] = rng.integers(0, 1 << 32, (3, (V + 31) // 32), dtype=np.uint64).astype(np.uint32) | np.uint32(0x10000001)
    res, _ = run_lean(c, 1, handed_back=1)
    assert res["exact"] == 3, res


@pytest.mark.parametrize("V,masked,n_hist", [(32000, False, 0), (50257, True, 300), (151936, False, 2000), (163844, True, 0), (262144, False, 700), (262144, True, 3000)])
def test_rows_whose_cut_no_list_holds(V, masked, n_hist):
    """Logits on a grid, thousands of tokens each step, the cut and the draw among them: answered by the exact path from what the sweep has left - with touched tokens
    in the ties and above them, before and behind the 16384th token, by top-p, min-p and both."""
    rows = 12
    c = _no_top_k(gc.make_cfg2(rows=rows, V=V, n_hist=n_hist, n_bias=50 if n_hist else 0))
    rng = np.random.default_rng(V)
    c["logits"] = (np.round(rng.standard_normal((rows, V)) * 4) / 2).astype(np.float32)
    c["inv_t"] = np.linspace(0.6, 1.2, rows).astype(np.float32)
    c["top_p"] = np.array([0.3, 0.5, 0.6, 0.7, 0.8, 0.9, 0.95, 0.99, 1.0, 1.0, 0.6, 0.9])
    c["min_p"] = np.array([0.0] * 8 + [0.02, 0.3, 0.05, 0.01])
    for r in range(rows):
        if n_hist:
            c["hist"][r][:2] = [V - 1, V - 1 - r % 4]
        c["logits"][r, V - 1 - r % 4] = 5.0
    if masked:
        on = rng.random((rows, (V + 31) // 32 * 32)) < 0.8
        c["allow"] = np.ascontiguousarray(np.packbits(on, axis=1, bitorder="little").view(np.uint32))
    res, smp = run_lean(c, 1, max_differ=1, handed_back=rows)
    fl, m = smp.flags.cpu().numpy(), gc.pkg()
    assert ((fl & m.FLAG_ROUTE_EXACT) != 0).sum() >= (1 if V < 100000 else 6), fl
    assert (((fl & m.FLAG_ROUTE_EXACT) != 0) <= ((fl & m.FLAG_ROUTE_HANDED_BACK) != 0)).all()
    nk = smp.n_kept.cpu().numpy()
    assert V < 100000 or (nk < 16384).any() and (nk > 16384).any()


@pytest.mark.parametrize("V", [50257, 163848, 200003])
@pytest.mark.parametrize("n_bias,named", [(2047, 2047), (2048, 2048), (3000, 2100)])
def test_more_bias_entries_than_the_batch_declares(V, n_bias, named):
    """Bias lists that fit max_hist + max_bias together, most of whose entries name one token, of the history too: it takes all of them, in their order, whatever
    room the count of a token's entries has in a kernel of those that batches with shorter lists get."""
    c = _no_top_k(gc.make_cfg2(rows=4, V=V, n_hist=4, n_bias=n_bias))
    c["inv_t"][:], c["top_p"][:], c["min_p"][:] = 1.0, 0.9, 0.0
    rng = np.random.default_rng(n_bias)
    for r in range(4):
        tok = V - 1 - 7 * r
        c["hist"][r][0] = tok
        c["bias_ids"][r, rng.permutation(n_bias)[:named]] = tok
        c["bias_vals"][r] = np.round(c["bias_vals"][r] * 64) / 65536  # (their sum lifts or lowers the token by some tenths)
        c["logits"][r, tok] = 7.0
    d = gc.upload(c, hints=True)
    d["max_hist"], d["max_bias"], d["min_p_min"] = 2500, 1000, 0.0
    smp = gc.sampler_for(c, d, 1, max_split=1).run()
    res = gc.compare_rows(c, smp, range(4), 1, check_kept=False)
    m, fl = gc.pkg(), smp.flags.cpu().numpy()
    assert res["differ"] == 0 and ((fl & (m.FLAG_ROUTE_LEAN | m.FLAG_ROUTE_HANDED_BACK)) != 0).all(), (res, fl)
    assert n_bias > 2047 or ((fl & m.FLAG_ROUTE_LEAN) != 0).all(), fl
