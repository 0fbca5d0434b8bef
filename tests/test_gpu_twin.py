"""GPU: short-list rows two a compute unit (ws_twin.h), which batches of more rows than compute units get, through the C ABI against the
CPU oracle on identical seeded inputs: vocabularies either side of a vector, of a chunk and of the sample, the tables behind the bitmap and
in the list's place, ids at hand and behind those, repeated bias entries, rows whose largest tokens lie far above the others, and the rows
left to the three-pass code. Bars as in test_gpu_short.py."""
import numpy as np
import pytest
import torch

import gpu_cases as gc
from test_gpu_short import _odd, run_short

pytestmark = pytest.mark.gpu


def rows_of():
    return torch.cuda.get_device_properties(0).multi_processor_count + 1


def some(rows, step=31):
    return sorted({0, 1, rows - 1, *range(0, rows, step)})


def twice_biased(c):
    """Every third row's first bias entries name one token three times, a token of its history."""
    for r in range(0, c["rows"], 3):
        c["bias_ids"][r, :3] = c["hist"][r, 0]
    return c


SIZES = [8, 9, 31, 2047, 2049, 8191, 16384, 16385, 16387, 18432, 18437, 20479, 50257]


@pytest.mark.parametrize("dtype,allowed", [("f32", None), ("f32", 0.3), ("bf16", None), ("bf16", 0.6)])
@pytest.mark.parametrize("V", SIZES)
def test_vocabularies_off_every_boundary(V, dtype, allowed):
    """Top-k rows and, every fourth, rows with a min-p alone (bf16: of the vocabularies that this kernel takes; ws_code.h has the others)."""
    rows = rows_of()
    c = _odd(rows, V, dtype, top_k=min(20, V), n_hist=min(300, V), n_bias=min(20, V), allowed=allowed)
    c["top_k"][::4] = 0
    c["min_p"][::4] = 0.02
    c["top_p"][1::4] = 1.0
    c["min_p"][2::4] = 0.1
    if allowed is not None:
        c["allow"][:, 0] |= 7  # (no row without a token)
    run_short(c if V < 300 else twice_biased(c), 1, rows=some(rows), handed_back=rows if V < 64 else 2)


@pytest.mark.parametrize("V,n_hist,n_bias,top_k,allowed", [(50257, 0, 0, 50, None), (50257, 0, 0, 50, 0.2), (50257, 1, 0, 3, None), (50257, 0, 1, 600, 0.5), (50257, 4608, 20, 50, None),
                                                           (50257, 4609, 0, 50, None), (40000, 9000, 1000, 200, None), (151936, 7000, 500, 1000, None), (262144, 8192, 500, 1000, 0.1),
                                                           (400000, 500, 20, 50, None)])
def test_histories_bias_lists_and_wide_top_k(V, n_hist, n_bias, top_k, allowed):
    """Tables of every size, a row's last ids at hand and the first behind them; one, two and eight candidates a thread."""
    rows = rows_of()
    c = _odd(rows, V, top_k=top_k, n_hist=max(n_hist, 1), n_bias=max(n_bias, 1), allowed=allowed)
    if not n_hist:
        c["hist"] = None
    if not n_bias:
        c["bias_ids"] = c["bias_vals"] = None
    c["top_p"][::2] = 1.0
    _, smp = run_short(c if n_hist == 0 or n_bias < 3 else twice_biased(c), 1, rows=some(rows, 67))
    was = [x.clone() for x in (smp.token, smp.n_kept, smp.stats, smp.kept_ids)]
    for _ in range(4):  # every row again: the same, whatever the two of a compute unit were at
        smp.kept_ids.fill_(-7)
        smp.run()
        assert torch.equal(was[0], smp.token) and torch.equal(was[1], smp.n_kept) and torch.equal(was[3], smp.kept_ids)
        assert torch.allclose(was[2], smp.stats, rtol=1e-6, atol=0)  # (the order of the sums differs)


@pytest.mark.parametrize("V,allowed", [(50257, None), (50259, 0.9)])
def test_min_p_rows_with_lists_of_thousands(V, allowed):
    """Floors that 1000 to 7000 tokens pass; many a row's sample puts its own floor too low for the list, and the row is listed again.
    Left to the three-pass code: rows whose list does not fit, and no others."""
    rows = rows_of()
    c = _odd(rows, V, top_k=0, min_p=0.0043, n_hist=200, n_bias=1, allowed=allowed)
    c["bias_ids"] = c["bias_vals"] = None
    c["logits"] = (np.random.default_rng(5).standard_normal((rows, V), dtype=np.float32) * 2).astype(np.float32)
    c["inv_t"][:] = 1.0
    c["hist"][:] = np.argpartition(c["logits"], 200, axis=1)[:, :200]  # (tokens that no list has)
    _, smp = run_short(c, 1, rows=some(rows), kept_cap=4096, handed_back=rows)
    x, m = c["logits"], gc.pkg()
    if allowed is not None:
        on = np.unpackbits(c["allow"].view(np.uint8), axis=1, bitorder="little")[:, :V].astype(bool)
        x = np.where(on, x, -np.inf)
    listed = (x > x.max(axis=1, keepdims=True) + np.log(0.0043)).sum(axis=1)
    back = (smp.flags.cpu().numpy() & m.FLAG_ROUTE_HANDED_BACK) != 0
    assert not back[listed < 3900].any() and back[listed > 4400].all()  # (0.02 e-folds more than the floor: a few per cent)
    assert (listed < 3900).sum() > rows // 4 and back.any()


@pytest.mark.parametrize("dtype,V,n_hist", [("f32", 100003, 64), ("bf16", 262144, 64), ("f32", 384961, 257), ("f32", 384930, 262), ("f32", 384930, 250)])
def test_rows_whose_largest_tokens_lie_far_above_the_others(dtype, V, n_hist):
    """Cold rows: a few tokens 58 to 76 units of the exponent above the rest; of most rows one or two are in the sample, of some none is. The counts of the
    sample's tokens reach their last bin, and are cleared again: tables of the touched tokens that would just not, and just, lie behind them in the list's place."""
    rows = rows_of()
    c = _odd(rows, V, dtype, top_k=50, n_hist=n_hist, n_bias=0)
    c["inv_t"][:] = 20.0
    rng = np.random.default_rng(rows)
    x = (rng.standard_normal((rows, V), dtype=np.float32) * 0.5)
    for r in range(rows):
        at = rng.integers(0, V, 6)
        if n_hist > 64:  # (touched tokens of the bitmap's first words, the first of the ranks)
            at[:3] = [31, 33, 70]
            c["hist"][r, 1:91] = np.arange(90)
        x[r, at] = (5.0 + 0.5 * rng.random()) + np.array([0.0, 0.013, 0.04, 0.11, 0.3, 0.4], np.float32)
        c["hist"][r, 0] = int(x[r].argmax())
    c["logits"] = gc.f32_to_bf16_bits(x) if dtype == "bf16" else x
    run_short(c, 1, rows=some(rows, 17), kept_cap=64, handed_back=rows // 50, top_k_max=50)


def test_rows_left_to_the_three_pass_code():
    """Rows that break the batch's word, rows of one value (more ties than the list holds), rows without a token, NaNs and infinities;
    the rows between them are the kernel's own."""
    rows, V = rows_of() + 300, 20001
    c = _odd(rows, V, top_k=40, n_hist=100, n_bias=0)
    c["top_k"][0] = 0
    c["top_k"][1] = 1025
    c["logits"][2:rows:50] = 1.5
    c["logits"][3, :] = -np.inf
    c["logits"][3, 77] = 0.25
    c["logits"][4, 100:200] = np.nan
    c["logits"][5, ::2] = -np.inf
    res, smp = run_short(c, 1, rows=list(range(10)) + some(rows), handed_back=rows, top_k_max=40)
    m = gc.pkg()
    back = (smp.flags.cpu().numpy() & m.FLAG_ROUTE_HANDED_BACK) != 0
    assert back[[0, 1, 3]].all() and back[2:rows:50].all()
    assert int(back.sum()) <= 5 + len(range(2, rows, 50)), np.flatnonzero(back)


def test_rows_with_bad_parameters_among_those_left_over():
    """The kernel behind takes several rows a workgroup: one with a bad temperature writes its flags at once, the rows after it - of the same workgroup,
    left over as well - are answered as ever."""
    cus = rows_of() - 1
    rows, V = 3 * cus, 20001
    c = _odd(rows, V, top_k=40, n_hist=100, n_bias=0)
    bad = np.arange(0, cus, 2)
    c["inv_t"][bad] = np.where(bad % 4, np.float32(-1), np.float32(0))
    c["top_k"][cus:] = 0  # (against the batch's word)
    m = gc.pkg()
    d = gc.upload(c, hints=True)
    d["top_k_max"] = 40
    for _ in range(3):
        smp = gc.sampler_for(c, d, 1).run()
        res = gc.compare_rows(c, smp, [1, 3, *range(cus, rows, 37), rows - 1], 1, check_kept=False)
        assert res["differ"] == 0, res
        fl = smp.flags.cpu().numpy()
        assert ((fl[bad] & m.FLAG_BAD_PARAM) != 0).all() and (smp.token.cpu().numpy()[bad] == -1).all()
        assert ((fl[cus:] & m.FLAG_ROUTE_HANDED_BACK) != 0).all() and not (fl[cus:] & m.FLAG_BAD_PARAM).any()


@pytest.mark.parametrize("V,top_k,n_hist,allowed", [(8192, 64, 0, None), (8193, 64, 0, None), (24576, 64, 1, None), (24577, 64, 300, None), (24576, 65, 300, 0.5), (16384, 128, 300, None),
                                                    (16385, 128, 1, 0.5), (12288, 256, 300, 0.5), (12289, 256, 300, None), (12288, 257, 300, None), (245760, 64, 300, None),
                                                    (245759, 64, 300, None), (245760, 128, 300, 0.3), (245760, 128, 300, None), (400000, 64, 300, 0.3)])
def test_bf16_rows_either_side_of_the_lines_between_the_kernels(V, top_k, n_hist, allowed):
    """Rows that go to this kernel or to ws_code.h by vocabulary, top-k, touched tokens and room: the answers are the oracle's on both sides."""
    rows = rows_of()
    c = _odd(rows, V, "bf16", top_k=top_k, n_hist=max(n_hist, 1), n_bias=0, allowed=allowed)
    if not n_hist:
        c["hist"] = None
    smp = gc.sampler_for(c, gc.upload(c, hints=True), 1).run()
    res = gc.compare_rows(c, smp, some(rows, 67), 1, check_kept=False)
    assert res["differ"] == 0 and res["exact"] == len(some(rows, 67)), res
    fl, m = smp.flags.cpu().numpy(), gc.pkg()
    assert (fl & m.FLAG_ROUTE_SHORT).all() and not (fl & m.FLAG_ROUTE_HANDED_BACK).any()


@pytest.mark.parametrize("V,n_hist,n_bias,allowed,dtype", [(50257, 2047, 0, 0.5, "f32"), (50257, 2048, 0, 0.5, "f32"), (50257, 2049, 0, 0.5, "f32"), (50257, 1500, 548, 0.5, "f32"),
                                                           (50257, 1500, 549, 0.5, "f32"), (12288, 2040, 8, 0.3, "bf16"), (262144, 8192, 500, 0.05, "f32"), (262144, 1542, 0, 0.5, "f32"),
                                                           (262144, 5, 3, 0.1, "f32")])
def test_masks_that_allow_the_whole_history(V, n_hist, n_bias, allowed, dtype):
    """The list of the entries that a mask allows, to its last place and past it: the mask allows few tokens, but of every other row all that its
    history and bias list name (so that more are listed than the mask let expect, and the row goes on without the list)."""
    rows = rows_of()
    c = _odd(rows, V, dtype, top_k=50, n_hist=n_hist, n_bias=max(n_bias, 1), allowed=allowed)
    for r in range(0, rows, 2):
        ids = np.concatenate([c["hist"][r], c["bias_ids"][r][:n_bias]]).astype(np.int64)
        ids = ids[(ids >= 0) & (ids < V)]
        np.bitwise_or.at(c["allow"][r], ids >> 5, (np.uint32(1) << (ids & 31).astype(np.uint32)).astype(c["allow"].dtype))
    if not n_bias:
        c["bias_ids"] = c["bias_vals"] = None
    run_short(c if n_bias < 3 else twice_biased(c), 1, rows=some(rows, 41))


@pytest.mark.parametrize("V,top_k,step,allowed", [(50257, 513, 0.0, None), (50257, 1024, 0.0, 0.5), (700, 700, 0.0, None), (1500, 1000, 0.0, None), (50257, 1000, 0.25, None), (50257, 1000, 0.004, None),
                                                  (262144, 1000, 0.0, 0.1)])
def test_wide_top_k_without_an_order(V, top_k, step, allowed):
    """A top-k of more than 512: cuts and draw by buckets - everything listed, more listed than kept, cuts by top-p, by min-p, by both and by neither; logits so
    coarse that a bucket is too full and the list is sorted after all, and just not so."""
    rows = rows_of()
    c = _odd(rows, V, top_k=top_k, n_hist=min(300, V), n_bias=min(20, V), allowed=allowed)
    if step:
        c["logits"] = (np.round(c["logits"] / step) * step).astype(np.float32)
    c["top_p"][::4] = 1.0
    c["top_p"][1::4] = 0.3
    c["min_p"][1::3] = 0.02
    c["min_p"][2::6] = 1.0
    c["inv_t"][::5] = 0.3
    run_short(c, 1, rows=some(rows, 23), handed_back=2)


# (The rows above are asked for a dump, and so they are sorted. The finish by buckets is for batches that ask for none.)
WIDE = [(50257, 513, 0.0, None), (50257, 1024, 0.0, 0.5), (700, 700, 0.0, None), (1500, 1000, 0.0, None), (50257, 1000, 0.25, None), (50257, 1000, 0.004, None), (262144, 1000, 0.0, 0.1)]


def _wide(rows, V, top_k, step, allowed):
    """Rows cut by top-k alone, by top-p (0.3 too), by min-p and by both, cold ones among them; step: the grid the logits lie on."""
    c = _odd(rows, V, top_k=top_k, n_hist=min(300, V), n_bias=min(20, V), allowed=allowed)
    if step:
        c["logits"] = (np.round(c["logits"] / step) * step).astype(np.float32)
    c["top_p"][::4] = 1.0
    c["top_p"][1::4] = 0.3
    c["min_p"][1::3] = 0.02
    c["min_p"][2::6] = 1.0
    c["inv_t"][::5] = 0.3
    return c


@pytest.mark.parametrize("V,top_k,step,allowed", WIDE)
def test_wide_top_k_by_buckets(V, top_k, step, allowed):
    """A top-k of more than 512 in a batch that asks for no dump, which is when cuts and draw go by buckets: everything listed, more listed than kept, cuts by
    top-p, by min-p, by both and by neither; logits so coarse that a bucket is too full and the list is sorted after all, and just not so."""
    rows = rows_of()
    c = _wide(rows, V, top_k, step, allowed)
    smp = gc.sampler_for(c, gc.upload(c, hints=True), 1, kept_cap=0).run()
    res = gc.compare_rows(c, smp, some(rows, 23), 1, check_kept=False)
    m, fl = gc.pkg(), smp.flags.cpu().numpy()
    short, back = (int(((fl & bit) != 0).sum()) for bit in (m.FLAG_ROUTE_SHORT, m.FLAG_ROUTE_HANDED_BACK))
    assert res["differ"] == 0 and short + back == rows and back <= 2, (res, short, back)


@pytest.mark.parametrize("V,top_k,step,allowed", WIDE)
def test_wide_top_k_by_buckets_and_by_the_sort(V, top_k, step, allowed):
    """The same rows with the dump, which are sorted: tokens, counts and flags are the same, and so are probabilities and distances to the decisions but for
    the rounding of 64-bit sums. A running mass of up to 2048 terms that reach it by chains of at most 30 additions is off by 30 x 2^-53 of itself on either side,
    a distance to a cut by that much of the cut's mass, which is what it is divided by: 8e-15, 1e-14 with the quotients' own roundings."""
    rows = rows_of()
    c = _wide(rows, V, top_k, step, allowed)
    got, want = (gc.sampler_for(c, gc.upload(c, hints=True), 1, kept_cap=cap).run() for cap in (0, 1024))
    m = gc.pkg()
    assert torch.equal(got.flags, want.flags)
    # (a min-p of 1 is the largest token's own mass: reported as near, and decided the same way)
    near = ((got.flags & m.FLAG_NEAR) != 0) & torch.from_numpy(c["min_p"] != 1.0).cuda()
    assert int(near.sum()) <= 2
    for k in ("token", "n_kept"):
        assert torch.equal(getattr(got, k)[~near], getattr(want, k)[~near]), k
    assert torch.allclose(got.prob, want.prob, rtol=3e-7, atol=0)  # (two roundings to 32 bits)
    # (a draw of the first or last token has 1e300 or 0 in the place of one distance on both sides)
    assert (got.margin - want.margin)[~near].abs().max().item() <= 1e-14


@pytest.mark.parametrize("V,n_bias,n_hist,allowed", [(262144, 4096, 3, 0.1), (262144, 5000, 1, 0.05), (50257, 4095, 4, 0.02), (50257, 6000, 2, 0.02), (50257, 4097, 0, 0.02)])
def test_masked_rows_with_more_bias_entries_than_the_batch_declares(V, n_bias, n_hist, allowed):
    """Lists that fit max_hist + max_bias together, of which the bias list is by far the longer one: a masked row takes each entry's own value, however many
    there are, and counts none as history."""
    rows = rows_of()
    c = _odd(rows, V, top_k=50, n_hist=max(n_hist, 1), n_bias=n_bias, allowed=allowed)
    if not n_hist:
        c["hist"] = np.full((rows, 1), -1, np.int32)
    for r in range(rows):  # (the last entries are allowed, and their tokens among the largest)
        ids = np.unique(c["bias_ids"][r, -40:]).astype(np.int64)
        np.bitwise_or.at(c["allow"][r], ids >> 5, (np.uint32(1) << (ids & 31).astype(np.uint32)).astype(c["allow"].dtype))
        c["logits"][r, ids[::2]] = 8.0
    d = gc.upload(c, hints=True)
    d["max_hist"], d["max_bias"] = 7700, 1000
    smp = gc.sampler_for(c, d, 1, kept_cap=1024).run()
    res = gc.compare_rows(c, smp, some(rows, 23), 1)
    m = gc.pkg()
    assert res["differ"] == 0 and (smp.flags.cpu().numpy() & m.FLAG_ROUTE_MASK == m.FLAG_ROUTE_SHORT).all(), res


@pytest.mark.parametrize("V,n_hist", [(50257, 0), (50260, 64), (262144, 8192), (384930, 262)])
def test_top_k_rows_whose_list_just_fits(V, n_hist):
    """Rows with 3840 to 4096 tokens above the threshold, all within a bin of it, spread over the row, in one stretch of it or in the last waves' share of every
    chunk: the list holds them, whatever places the waves had taken. With one more it does not."""
    rows = rows_of()
    c = _odd(rows, V, top_k=1000, n_hist=max(n_hist, 1), n_bias=0)
    c["bias_ids"] = c["bias_vals"] = None
    rng = np.random.default_rng(V)
    c["logits"][:] = (rng.standard_normal((rows, V), dtype=np.float32) - 30).astype(np.float32)
    c["inv_t"][:], c["top_p"][:], c["min_p"][:] = 1.0, 0.95, 0.0
    if not n_hist:
        c["hist"] = None
    listed = np.array([3840, 3849, 3900, 4000, 4064, 4090, 4095, 4096, 4097, 4200])[np.arange(rows) % 10]
    for r in range(rows):
        kind = r // 10 % 3
        if kind == 0:
            at = rng.permutation(V)[:listed[r]]
        elif kind == 1:
            at = rng.integers(0, V - listed[r]) + np.arange(listed[r])
        else:
            at = np.flatnonzero(np.arange(V) % 2048 >= 1536)
            at = at[rng.permutation(at.size)[:listed[r]]]
        if n_hist:  # (none of them touched)
            c["hist"][r] = rng.permutation(np.setdiff1d(np.arange(20000), at))[:n_hist]
        c["logits"][r, at] = 2.0 + rng.uniform(0.0, 0.028, at.size).astype(np.float32)
    _, smp = run_short(c, 1, rows=some(rows), handed_back=rows)
    back = (smp.flags.cpu().numpy() & gc.pkg().FLAG_ROUTE_HANDED_BACK) != 0
    # (a stretch that the sample misses puts the threshold far below, where everything is listed)
    sampled = np.arange(rows) // 10 % 3 != 1
    assert not back[(listed <= 4096) & sampled].any(), listed[back & (listed <= 4096) & sampled]
    assert back[listed > 4096].all()


@pytest.mark.parametrize("V,dtype,n_hist", [(16384, "f32", 0), (20483, "f32", 40), (50260, "f32", 700), (33001, "bf16", 0), (12289, "bf16", 64)])
def test_lists_of_few_places(V, dtype, n_hist):
    """Rows whose list takes up to 512 places, a few more or many more, by a min-p alone or a small top-k: tokens spread over the row, in one wave's share of every
    chunk, in one vector, in the tokens behind the last vector."""
    rows = rows_of()
    c = _odd(rows, V, top_k=0, n_hist=max(n_hist, 1), n_bias=0)
    c["bias_ids"] = c["bias_vals"] = None
    if not n_hist:
        c["hist"] = None
    rng = np.random.default_rng(V)
    x = (rng.standard_normal((rows, V), dtype=np.float32) - 30).astype(np.float32)
    c["inv_t"][:], c["top_p"][:], c["min_p"][:] = 1.0, 0.95, 0.05
    listed = np.array([1, 2, 8, 31, 32, 33, 63, 64, 65, 127, 129, 250, 256, 257, 300, 400, 480, 511, 513, 700])[np.arange(rows) % 20]
    for r in range(rows):
        kind = r // 20 % 4
        if kind == 0:
            at = rng.permutation(V)[:listed[r]]
        elif kind == 1:
            at = np.flatnonzero(np.arange(V) % 2048 < 256)
            at = at[rng.permutation(at.size)[:listed[r]]]
        elif kind == 2:
            at = rng.integers(0, V - listed[r]) + np.arange(listed[r])
        else:
            at = V - 1 - np.arange(listed[r])
        if n_hist:
            c["hist"][r][:min(5, at.size)] = at[:5]  # (a few of them touched)
        x[r, at] = 4.0 + rng.uniform(0.0, 2.5, at.size).astype(np.float32)
    c["logits"] = x
    if dtype == "bf16":
        c["logits"], c["dtype"] = gc.f32_to_bf16_bits(x), "bf16"
    run_short(c, 1, rows=some(rows, 3), handed_back=1)
    c["top_k"][:] = 8
    c["min_p"][:] = 0.0
    run_short(c, 1, rows=some(rows, 7), handed_back=1)


@pytest.mark.parametrize("n_hist,n_bias", [(2040, 8), (2040, 9), (1, 2047), (2, 2047), (2048, 0), (2049, 0)])
@pytest.mark.parametrize("V,allowed,dtype", [(9792, 0.05, "f32"), (50257, 0.3, "bf16")])
def test_masked_rows_at_the_length_from_which_allowed_entries_are_listed(V, allowed, dtype, n_hist, n_bias):
    """Lists of 2048 entries and of one more, with tokens that several bias entries name."""
    rows = rows_of()
    c = _odd(rows, V, dtype, top_k=30, n_hist=n_hist, n_bias=n_bias, allowed=allowed)
    if not n_bias:
        c["bias_ids"] = c["bias_vals"] = None
    run_short(c if n_bias < 3 else twice_biased(c), 1, rows=some(rows, 41), handed_back=1)
