"""GPU: short-list rows shared between workgroups that hold them in registers (ws_few.h), through the C ABI against the CPU
oracle on identical seeded inputs, at the sizes where its split can go wrong: vocabularies one token either side of a vector,
of a chunk and of a share, rows off every alignment, the longest history it takes, tokens with several bias entries, ties at
the threshold, rows it has to hand back. Bars as in test_gpu_sample.py (gpu_cases.compare_rows)."""
import numpy as np
import pytest
import torch

import gpu_cases as gc

pytestmark = pytest.mark.gpu


def case(rows, V, dtype="f32", top_k=40, min_p=0.0, n_hist=300, n_bias=20, allowed=None, seed=3):
    c = gc.make_cfg2(rows=rows, V=V, n_hist=n_hist, n_bias=n_bias)
    rng = np.random.default_rng(seed)
    c["top_k"][:] = top_k
    c["min_p"][:] = min_p
    if dtype == "bf16":
        c["logits"], c["dtype"] = gc.f32_to_bf16_bits(c["logits"]), "bf16"
    if allowed is not None:
        words = (V + 31) // 32
        c["allow"] = np.ascontiguousarray(np.packbits(rng.random((rows, words * 32)) < allowed, axis=1, bitorder="little").view(np.uint32))
    return c


def run(c, handed_back=0, max_differ=0, max_split=0, **more):
    m = gc.pkg()
    d = gc.upload(c, hints=True, min_p_hint=True)
    smp = gc.sampler_for(c, d, 1, kept_cap=1024, max_split=max_split, **more)
    assert m.lib().ws_sample_batch_workspace_use(smp.desc) == m.WORK_MEETING  # (the rows are shared)
    for _ in range(2):  # the second launch finds the workspace as the first left it
        smp.run()
    res = gc.compare_rows(c, smp, range(c["rows"]), 1)
    assert res["differ"] <= max_differ and res["exact"] + res["differ"] == c["rows"], res
    fl = smp.flags.cpu().numpy()
    back = int(((fl & m.FLAG_ROUTE_HANDED_BACK) != 0).sum())
    assert back <= handed_back and int(((fl & m.FLAG_ROUTE_SHORT) != 0).sum()) + back == c["rows"], fl
    assert not smp.workspace.any().item(), "the workspace is not zero after the launch"
    return smp


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V", [4097, 8191, 8200, 32771, 50257, 65535, 151935, 151937])
def test_vocabularies_off_every_boundary(V, dtype):
    run(case(3, V, dtype))


@pytest.mark.parametrize("max_split", [2, 3, 4, 7, 16])
def test_any_number_of_parts(max_split):
    """Parts that are no power of two; two parts of 40960 tokens, the most a workgroup holds."""
    run(case(2, 81920, top_k=50), max_split=max_split)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V,max_split", [(81921, 2), (114681, 2), (114688, 2), (172032, 3), (172025, 3)])
def test_shares_of_112_tokens_a_thread(V, max_split, dtype):
    """Too few parts for shares of 80 tokens a thread: the smallest and the largest rows of the wide ones."""
    run(case(2, V, dtype, top_k=50, n_hist=1500, allowed=0.7 if V % 2 else None), max_split=max_split)


@pytest.mark.parametrize("dtype,top_k", [("f32", 1), ("f32", 512), ("bf16", 513), ("f32", 1024), ("bf16", 64)])
def test_top_k_from_one_to_the_largest(dtype, top_k):
    run(case(2, 40003, dtype, top_k=top_k), max_differ=1 if dtype == "bf16" else 0)


@pytest.mark.parametrize("dtype,allowed", [("f32", 0.1), ("bf16", 0.5)])
def test_rows_with_an_allow_mask(dtype, allowed):
    run(case(3, 33001, dtype, allowed=allowed))


@pytest.mark.parametrize("min_p", [1.0, 0.2, 0.05])
def test_min_p_without_a_top_k(min_p):
    run(case(4, 60001, top_k=0, min_p=min_p), max_differ=1, handed_back=1 if min_p < 0.1 else 0)


@pytest.mark.parametrize("dtype,rows,V,slots,chunk", [("f32", 16, 32768, 59, 32), ("bf16", 16, 32768, 59, 64), ("f32", 127, 16384, 478, 32), ("f32", 16, 32769, 59, 128)])
def test_a_waves_list_holds_what_the_header_says(dtype, rows, V, slots, chunk):
    """Min-p rows of sixteen and of two parts whose floor lets through tokens of one wave's share alone: as many as the wave lists
    at most, and one more, which hands the row back. Answers are the oracle's either way."""
    m = gc.pkg()
    rng = np.random.default_rng(slots)
    c = case(rows, V, top_k=0, min_p=0.5, n_hist=0, n_bias=0)
    waves = 8 * (16 if rows == 16 else 2)
    ids = np.concatenate([np.arange(chunk) + chunk * (5 + waves * k) for k in range(1 + (slots + 1) // chunk)])  # of the wave 5 of the row
    c["logits"][:] = -50.0 - 1e4 * rng.random((rows, V), dtype=np.float32)  # (far apart: no part lists more than a few of these)
    c["inv_t"][:] = 1.0
    c["top_p"][:] = 1.0
    for r in range(rows):
        n = slots + (r & 1)
        c["logits"][r, rng.permutation(ids)[:n]] = rng.permutation(n).astype(np.float32) / (2 * n)  # (a floor of half lets 0.69 units through)
    if dtype == "bf16":
        c["logits"], c["dtype"] = gc.f32_to_bf16_bits(c["logits"]), "bf16"
    d = gc.upload(c, hints=True, min_p_hint=True)
    smp = gc.sampler_for(c, d, 1, kept_cap=1024)
    for _ in range(2):
        smp.run()
    res = gc.compare_rows(c, smp, range(0, rows, 1 if rows == 16 else 9), 1)
    assert res["differ"] == 0, res
    back = (smp.flags.cpu().numpy() & m.FLAG_ROUTE_HANDED_BACK) != 0
    assert np.array_equal(back, np.arange(rows) % 2 == 1), back
    assert not smp.workspace.any().item()


def test_long_histories_and_repeated_bias_entries():
    """9000 ids of few tokens, so that counts are in the hundreds, and bias lists that name tokens of the history, some of
    them three times (their values are added in the order of the list)."""
    c = case(2, 90001, n_hist=9000, n_bias=60)
    c["hist"] %= 700
    c["bias_ids"][:, 20:40] = c["bias_ids"][:, :20]
    c["bias_ids"][:, 40:50] = c["bias_ids"][:, :10]
    c["bias_ids"][:, 50:] = c["hist"][:, :10]
    run(c)


def test_ties_at_the_threshold_and_a_row_of_one_value():
    """Logits rounded to halves: the threshold falls among ties; more of them than a wave lists, and the row is handed back.
    A row of equal logits is handed back as well and still the oracle's."""
    c = case(4, 30000, top_k=20, n_hist=0, n_bias=0)
    c["logits"][:2] = np.round(c["logits"][:2] * 2) / 2
    c["logits"][3] = 1.25
    run(c, handed_back=3)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V,masked,by_p", [(32771, False, False), (50257, True, False), (32768, False, True), (151937, True, True)])
def test_nan_of_either_kind_and_infinities_are_no_candidates(V, masked, by_p, dtype):
    """NaN, quiet and signalling, of either sign: in the vectors of the row's largest tokens, on tokens that the lists name, all over a wave's chunk and at
    the row's end; -inf in between, also at named tokens; and +inf under the mask. All of them count for -inf, none hands its row back."""
    c = case(3, V, dtype, top_k=0 if by_p else 40, min_p=0.3 if by_p else 0.0, n_hist=900, n_bias=64, allowed=0.5 if masked else None)
    rng = np.random.default_rng(V)
    bits = c["logits"].view(np.uint32 if dtype == "f32" else np.uint16)
    sh, per = (16, 4) if dtype == "f32" else (0, 8)
    quiet, signalling, low = 0x7FC0 << sh, 0x7F81 << sh, 0xFF80 << sh
    one_bit = signalling if dtype == "bf16" else 0x7F800001  # (a signalling NaN whose only set bit is the last)
    kinds = np.array([quiet, quiet | 0x8000 << sh, signalling, signalling | 0x8000 << sh, one_bit, low], dtype=bits.dtype)
    c["bias_vals"][:] = np.minimum(c["bias_vals"], 1.0)
    for r in range(3):
        top = np.argsort(gc.row_f32(c, r))[-60:]
        beside = top[top // per * per + (top + 1) % per < V]
        beside = beside // per * per + (beside + 1) % per  # another token of the vector
        named = np.concatenate([c["hist"][r][::5], c["bias_ids"][r][::3]])
        chunk = np.arange(7 * 8 * per, 15 * 8 * per)  # whole chunks of eight lanes: a wave's only vectors in a load
        spoilt = np.concatenate([np.setdiff1d(beside, top[-50:]), named, chunk, rng.integers(0, V, 300), [V - 1 - r, V - 2 - r]])
        bits[r, spoilt] = kinds[rng.integers(0, kinds.size, spoilt.size)]
        if masked:
            out = np.flatnonzero(~np.unpackbits(c["allow"][r].view(np.uint8), bitorder="little")[:V].astype(bool))
            bits[r, out[rng.integers(0, out.size, 40)]] = 0x7F80 << sh
            bits[r, np.intersect1d(out, c["hist"][r])[:5]] = 0x7F80 << sh
    run(c, max_differ=1 if dtype == "bf16" else 0)


@pytest.mark.parametrize("inv_t", [0.7, 1.25])
def test_the_waves_sums_meet_in_64_bits(inv_t):
    """128 tokens, every one a different wave's only one (a wave's own sum is exactly one), so that the normaliser is made of the
    factors that bring the waves' sums to the row's maximum: it has to be the 64-bit sum, rounded once."""
    m = gc.pkg()
    rng = np.random.default_rng(17)
    rows, V = 16, 32768  # sixteen parts a row, chunks of 32 tokens dealt to 128 waves
    x = np.full((rows, V), -np.inf, np.float32)
    at = 32 * np.arange(128) + rng.integers(0, 32, (rows, 128))
    np.put_along_axis(x, at, rng.uniform(0.0, 9.0, (rows, 128)).astype(np.float32), 1)
    d = [torch.full((rows,), v, dtype=dt, device="cuda") for v, dt in ((inv_t, torch.float32), (7, torch.int64), (0, torch.int64), (40, torch.int32))]
    smp = m.BatchSampler(torch.from_numpy(x).cuda(), d[0], d[1], d[2], top_k=d[3], top_k_max=40).run()
    got = smp.stats.cpu().numpy()
    assert (smp.flags.cpu().numpy() & m.FLAG_ROUTE_MASK == m.FLAG_ROUTE_SHORT).all()
    top = x.max(axis=1)
    want = np.exp((x - top[:, None]).astype(np.float64) * np.float64(np.float32(inv_t))).sum(axis=1)
    assert np.array_equal(got[:, 0], top)
    # (a rounding of the 64-bit sum to 32 bits differs between two orders of it once in 2^24 or so)
    assert np.array_equal(got[:, 1], want.astype(np.float32)), (got[:, 1] - want.astype(np.float32)) / want


def test_query_and_entropy():
    """Probability of a named token and the kept set's entropy from the sorted candidates."""
    m = gc.pkg()
    c = case(6, 32003, top_k=40)
    want = [gc.oracle_row(c, r, 1) for r in range(6)]
    query = np.array([w[1]["id"][r % 2] for r, w in enumerate(want)], np.int32)
    query[4] = np.setdiff1d(np.arange(c["V"]), want[4][1]["id"])[0]
    query[5] = -1
    smp = run(c, query=torch.from_numpy(query).cuda(), want_entropy=True)
    qp, ent = smp.query_prob.cpu().numpy(), smp.entropy.cpu().numpy()
    for r, (o, kept, _) in enumerate(want):
        hit = kept["p"][kept["id"] == query[r]]
        p_want = float(hit[0]) if hit.size else 0.0
        assert abs(qp[r] - p_want) <= 1e-6 * max(p_want, 1e-300), (r, qp[r], p_want)  # the bar of the token's probability
        pk = kept["p"][kept["p"] > 0]
        h_want = float(-(pk * np.log(pk)).sum())
        assert abs(ent[r] - h_want) <= 1e-6 * max(1.0, h_want), (r, ent[r], h_want)
    assert not (smp.flags.cpu().numpy() & m.FLAG_APPROX_ENTROPY).any()


@pytest.mark.parametrize("rows,n,K", [(2, 32768, 512), (100, 81920, 40), (5, 163844, 300), (1, 655360, 64), (16, 100000, 17)])
def test_top_lists_at_the_edges_of_a_share(rows, n, K):
    """ws_topk_rows_ws and ws_dflash_topk_ws (ws_top.h) with the smallest and the largest shares: ids, values and maxima equal to
    those of the kernels that give a row to one workgroup, twice on one workspace, which is zero again afterwards."""
    m = gc.pkg()
    rng = np.random.default_rng(n)
    x = torch.from_numpy((rng.standard_normal((rows, n)) * 2).astype(np.float32)).cuda()
    work = m.topk_rows_workspace(n, K, rows)
    want = m.topk_rows(x, K, 1.25)
    k = min(K, 64)
    first = m.dflash_topk(x, k)
    for _ in range(2):
        got = m.topk_rows(x, K, 1.25, workspace=work)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and torch.equal(got[2][:, 0], want[2][:, 0])
        assert torch.allclose(got[2][:, 1], want[2][:, 1], rtol=2e-6, atol=0)  # (float sums in another order: the bar of ws_topk_rows_ws)
        again = m.dflash_topk(x, k, workspace=work)
        assert torch.equal(again[0], first[0]) and torch.equal(again[1], first[1])
    assert not work.any().item()


@pytest.mark.parametrize("rows,n", [(1, 8191), (1, 8192), (3, 12289), (32, 50257), (127, 8200), (128, 9001), (129, 8195)])
def test_greedy_picks_shared_between_workgroups(rows, n):
    """Vocabularies and row counts either side of the rule that shares a row, ties across its parts, a row of one value, a row
    of -inf: the lowest index of the largest logit, on the current stream, on others, and twice on each."""
    m = gc.pkg()
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((rows, n)) * 2).astype(np.float32)
    for r in range(rows):
        x[r, rng.integers(0, n, 3)] = 50.0
    x[0], x[rows - 1, :] = 1.5, (-np.inf if rows > 1 else 1.5)
    x[rows // 2, n - 1] = 60.0 if rows > 2 else x[rows // 2, n - 1]
    want = x.argmax(axis=1)
    d = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    for stream in [torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()]:
        with torch.cuda.stream(stream):
            for _ in range(2):
                got = m.argmax_rows(d)
                to = torch.full((40,), -7, dtype=torch.int32, device="cuda")
                if rows <= 32:
                    m.argmax_rows_to(d, to, list(range(rows, 0, -1)))
                ids, pos = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.full((1,), 5, dtype=torch.int32, device="cuda")
                one = m.argmax(d[rows - 1], ids, pos, 2)
                stream.synchronize()
                assert np.array_equal(got.cpu().numpy(), want)
                assert rows > 32 or np.array_equal(to.cpu().numpy()[1:rows + 1][::-1], want)
                assert one.item() == ids.item() == want[rows - 1] and pos.item() == 7


def test_greedy_picks_over_any_workspace_and_under_capture():
    """The picks' workspace may hold anything when a launch begins - what the allocator left there, a launch of another shape, the
    launch's own words of an earlier replay -, a stream beyond the 64th has the same kernel as the first, and so has a captured
    one: replays over other logits, with other work on the memory between them, give every replay's picks."""
    m = gc.pkg()
    L = m.lib()
    rng = np.random.default_rng(5)
    rows, n = 8, 50257
    xs = [torch.from_numpy((rng.standard_normal((rows, n)) * 2).astype(np.float32)).cuda() for _ in range(3)]
    want = [x.argmax(dim=1).to(torch.int32) for x in xs]
    need = int(L.ws_argmax_workspace(n, rows))
    assert 0 < need <= 4096 and int(L.ws_argmax_workspace(4096, rows)) == 0
    out = torch.empty(rows, dtype=torch.int32, device="cuda")
    work = torch.empty(need // 8, dtype=torch.int64, device="cuda")

    def pick(x, out, work, stream):
        m.check(L.ws_argmax_rows_ws(stream, x.data_ptr(), n, out.data_ptr(), rows, work.data_ptr(), need), "ws_argmax_rows_ws")

    here = torch.cuda.current_stream().cuda_stream
    for k, fill in enumerate([0, -1, 0x7fffffffffffffff, None, None]):
        if fill is not None:
            work.fill_(fill)
        elif k == 3:
            work.copy_(torch.from_numpy(rng.integers(-2**62, 2**62, need // 8)))
        pick(xs[k % 3], out, work, here)
        assert torch.equal(out, want[k % 3]), k
    for k in range(70):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got = m.argmax_rows(xs[k % 3])
        s.synchronize()
        assert torch.equal(got, want[k % 3])

    x = xs[0].clone()
    ids, pos = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        g.capture_begin()
        got, one = m.argmax_rows(x), m.argmax(x[3], ids, pos, 1)
        g.capture_end()
        for k in range(6):
            x.copy_(xs[k % 3])
            g.replay()
            side.synchronize()
            assert torch.equal(got, want[k % 3]) and one.item() == ids.item() == want[k % 3][3].item() and pos.item() == k + 1, k
    # without a workspace, or with too little of it: the kernel that gives a row to one workgroup
    for w, b in ((None, 0), (work.data_ptr(), need - 1), (work.data_ptr() + 4, need)):
        out.fill_(-1)
        m.check(L.ws_argmax_rows_ws(here, xs[1].data_ptr(), n, out.data_ptr(), rows, w, b), "ws_argmax_rows_ws")
        assert torch.equal(out, want[1])


def test_greedy_pick_of_a_row_beyond_32_bit_offsets():
    """2^30 + 12 tokens, the largest of them behind byte 2^32 of the row."""
    m = gc.pkg()
    n = (1 << 30) + 12
    x = torch.zeros(n, dtype=torch.float32, device="cuda")
    x[n - 5] = 1.0
    x[7] = 0.5  # (where an offset that lost its 33rd bit would look)
    ids, pos = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    assert m.argmax(x, ids, pos).item() == ids.item() == n - 5
    assert m.argmax_rows(x.view(1, n)).item() == n - 5


@pytest.mark.parametrize("rows,top_k", [(1, 40), (5, 40), (200, 40), (3, 0)])
def test_notify_writes_its_words_once_the_results_are_in_host_memory(rows, top_k):
    """ws_sample_batch_notify on rows the registers kernel takes (it writes the words itself), on rows with a workgroup each and on
    rows without a top-k (the stream does): all words come, and then tokens and kept sets in pinned memory are the eager call's."""
    import time
    m = gc.pkg()
    c = case(rows, 40003 if top_k else 40000, top_k=top_k)
    d = gc.upload(c, hints=top_k > 0)
    want = gc.sampler_for(c, d, 1, kept_cap=64).run()
    torch.cuda.synchronize()
    smp = gc.sampler_for(c, d, 1, kept_cap=64)
    host = dict(token=torch.zeros(rows, dtype=torch.int32, pin_memory=True), n_kept=torch.zeros(rows, dtype=torch.int32, pin_memory=True),
                kept_ids=torch.full((rows, 64), -1, dtype=torch.int32, pin_memory=True))
    smp.desc.token, smp.desc.n_kept, smp.desc.kept_ids = (host[k].data_ptr() for k in ("token", "n_kept", "kept_ids"))
    done = torch.zeros(rows, dtype=torch.int32, pin_memory=True)
    words = done.numpy()
    for turn in (1, 2, 7):
        host["token"].fill_(-5)
        m.check(m.lib().ws_sample_batch_notify(torch.cuda.current_stream().cuda_stream, m.C.byref(smp.desc), done.data_ptr(), turn), "ws_sample_batch_notify")
        until = time.monotonic() + 20.0
        while not (words == turn).all() and time.monotonic() < until:
            pass
        assert (words == turn).all(), words
        assert torch.equal(host["token"], want.token.cpu()) and torch.equal(host["n_kept"], want.n_kept.cpu())
        assert torch.equal(host["kept_ids"], want.kept_ids.cpu())
    torch.cuda.synchronize()
    assert m.lib().ws_sample_batch_notify(None, m.C.byref(smp.desc), None, 1) == -1


def test_one_workspace_for_batches_of_any_shape():
    """Small and large vocabularies, many and few parts, the kernel that holds rows in registers, the short-list kernel's slices and
    the single sweep's parts, one after the other on one workspace that was cleared once: answers as on one of their own."""
    m = gc.pkg()
    work = torch.zeros(128 * 65792, dtype=torch.uint8, device="cuda")
    shapes = [(2, 4097, 5, "f32"), (1, 151936, 40, "f32"), (90, 131072, 30, "f32"), (3, 8192, 1000, "bf16"), (3, 65536, 0, "f32"), (60, 20000, 20, "bf16"),
              (1, 262144, 64, "bf16"), (16, 151936, 0, "f32"), (2, 100003, 513, "f32")]
    for rows, V, top_k, dtype in shapes + shapes[::-1]:
        c = case(rows, V, dtype, top_k=top_k)
        d = gc.upload(c, hints=top_k > 0)
        smp = gc.sampler_for(c, d, 1, kept_cap=0)
        assert smp.workspace.numel() <= work.numel()
        want = smp.run()
        got = gc.sampler_for(c, d, 1, kept_cap=0)
        got.desc.workspace, got.desc.workspace_bytes = work.data_ptr(), work.numel()
        got.run()
        torch.cuda.synchronize()
        assert torch.equal(got.token, want.token) and torch.equal(got.n_kept, want.n_kept) and torch.equal(got.flags, want.flags), (rows, V, top_k)
        assert torch.allclose(got.stats, want.stats, rtol=1e-6, atol=0)  # (a shared row's sum is taken in the order its parts arrive)
        assert not work.any().item(), (rows, V, top_k)


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 16, 17, 33])
def test_rows_whose_parts_share_a_chiplet_and_rows_whose_parts_do_not(rows):
    """Up to 16 rows of 16 parts go a row to a chiplet, with workgroups that have no row where the rows are no multiple of eight; 17 and 33 do not."""
    run(case(rows, 32771, n_hist=200, n_bias=5))
    m = gc.pkg()
    x = torch.from_numpy((np.random.default_rng(rows).standard_normal((rows, 32772)) * 2).astype(np.float32)).cuda()
    work = m.topk_rows_workspace(32772, 64, rows)
    for _ in range(2):
        got = m.topk_rows(x, 64, 1.0, workspace=work)
        assert torch.equal(got[0], m.topk_rows(x, 64, 1.0)[0]) and not work.any().item()


@pytest.mark.parametrize("kind", ["normal", "steps", "halves", "far", "flat"])
@pytest.mark.parametrize("K", [129, 300, 512])
def test_top_lists_whose_last_bucket_alone_is_put_in_order(kind, K):
    """Lists of more than 128 keys: distinct logits, many ties at the cut, most of the row tied, one token so far above the others that
    they share a bucket, and a row of one value."""
    m = gc.pkg()
    x = (np.random.default_rng(K).standard_normal((3, 40000)) * 2).astype(np.float32)
    if kind in ("steps", "halves"):
        x = np.round(x * (32 if kind == "steps" else 2)) / np.float32(32 if kind == "steps" else 2)
    if kind == "far":
        x[:, 777] = 1e30
    if kind == "flat":
        x[:] = 0.25
    dx = torch.from_numpy(x).cuda()
    work = m.topk_rows_workspace(x.shape[1], K, x.shape[0])
    for _ in range(2):
        ids, vals, _ = m.topk_rows(dx, K, 1.25, workspace=work)
        for r in range(x.shape[0]):
            want = np.sort(np.lexsort((np.arange(x.shape[1]), -x[r].astype(np.float64)))[:K])
            assert np.array_equal(ids[r].cpu().numpy(), want) and np.array_equal(vals[r].cpu().numpy(), x[r][want])
    assert not work.any().item()


@pytest.mark.parametrize("n", [4096, 8003, 24064, 34298])
def test_draft_draws_of_rows_of_any_length_are_shared(n):
    """ws_draft_sample_rows_ws against the kernel that gives a row to one workgroup, with and without a vocabulary map, for every number of
    candidates a step of its sums can end at: same candidates, draws and probabilities (the normaliser: float sums in another order)."""
    m = gc.pkg()
    rng = np.random.default_rng(n)
    tks = [1, 3, 4, 5, 20, 31, 32, 0, 40]
    rows = len(tks)
    x = torch.from_numpy((rng.standard_normal((rows, n)) * 3).astype(np.float32)).cuda()
    vmap = torch.from_numpy(rng.permutation(n).astype(np.int32)).cuda()
    work = torch.zeros(int(m.lib().ws_draft_sample_rows_workspace(n, rows)), dtype=torch.uint8, device="cuda")
    assert work.numel() > 0
    args = [dict(top_k=tks[b], qoff=b * m.Q_WORDS, inv_t=1.1, top_p=[1.0, 0.95, 0.6][b % 3], min_p=[0.0, 0.02][b % 2], key=int(rng.integers(1, 1 << 62))) for b in range(rows)]
    for mp in (None, vmap):
        got = []
        for w in (None, work):
            ctl = torch.zeros(rows * 64, dtype=torch.int32, device="cuda")
            q = torch.zeros(rows * m.Q_WORDS, dtype=torch.int32, device="cuda")
            m.draft_sample_rows(x, ctl, [64 * b for b in range(rows)], 2, args, q, vmap=mp, workspace=w)
            got.append((ctl.cpu(), q.cpu().view(rows, m.Q_WORDS)))
        (c0, q0), (c1, q1) = got
        assert torch.equal(c0, c1) and torch.equal(q0[:, :33], q1[:, :33])
        assert torch.allclose(q0[:, 33:65].contiguous().view(torch.float32), q1[:, 33:65].contiguous().view(torch.float32), rtol=1e-5, atol=1e-9)
    assert not work.any().item()
