"""GPU: a lone row whose parameters and history ids travel with the launch (ws_sample_batch_notify_host) against the same row read from memory
(ws_sample_batch): the same kernel otherwise, so every answer is the same, bit for bit. History lengths on both sides of what fits the
arguments; rows without a history, with a bias list, with a min-p in the top-k's place; rows the launch does another way."""
import time

import numpy as np
import pytest
import torch

import gpu_cases as gc

pytestmark = pytest.mark.gpu


def pinned(a):
    t = torch.empty(a.shape, dtype=torch.from_numpy(a).dtype, pin_memory=True)
    t.copy_(torch.from_numpy(a))
    return t


@pytest.mark.parametrize("vocab,top_k,min_p,n_hist,declared,n_bias,rows", [
    (151936, 40, 0.0, 256, 256, 0, 1), (151936, 40, 0.0, 0, 0, 0, 1), (151936, 40, 0.05, 1, 4, 3, 1), (50257, 7, 0.0, 767, 768, 0, 1),
    (50257, 40, 0.0, 768, 768, 70, 1), (50257, 40, 0.0, 769, 800, 0, 1), (262144, 300, 0.0, 511, 511, 0, 1), (40003, 0, 0.1, 300, 300, 9, 1),
    (19471, 40, 0.0, 958, 958, 0, 1), (19471, 40, 0.0, 40, 12, 0, 1), (40003, 0, 0.0, 100, 100, 0, 1), (40003, 40, 0.0, 64, 64, 0, 3)])
def test_the_row_of_the_arguments_is_the_row_of_memory(vocab, top_k, min_p, n_hist, declared, n_bias, rows):
    m = gc.pkg()
    rng = np.random.default_rng(vocab + n_hist)
    x = torch.from_numpy(rng.normal(0, 2, (rows, vocab)).astype(np.float32)).cuda()
    args = dict(inv_t=np.full(rows, 1.25, np.float32), top_p=np.full(rows, 0.95), min_p=np.full(rows, min_p), seed=np.arange(rows, dtype=np.int64) + (77 << 33),
                step=np.arange(rows, dtype=np.int64) + 5, top_k=np.full(rows, top_k, np.int32))
    hints = dict(top_k_max=top_k, min_p_min=min_p if not top_k and min_p else 0.0)
    if n_hist:
        args.update(hist=(rng.random(n_hist * rows) ** 2 * vocab).astype(np.int32), hist_off=np.arange(rows + 1, dtype=np.int32) * n_hist,
                    rep=np.full(rows, 1.3, np.float32), pres=np.full(rows, 0.3, np.float32), freq=np.full(rows, 0.02, np.float32))
        hints.update(max_hist=declared)
    if n_bias:
        args.update(bias_ids=rng.integers(0, vocab, n_bias * rows).astype(np.int32), bias_vals=rng.normal(0, 3, n_bias * rows).astype(np.float32),
                    bias_off=np.arange(rows + 1, dtype=np.int32) * n_bias)
        hints.update(max_bias=n_bias)
    args = {k: pinned(v) for k, v in args.items()}
    make = lambda: m.BatchSampler(x, args["inv_t"], args["seed"], args["step"], kept_cap=512, **hints, **{k: v for k, v in args.items() if k not in ("inv_t", "seed", "step")})
    want, got = make().run(), make()
    torch.cuda.synchronize()
    done = torch.zeros(rows, dtype=torch.int32, pin_memory=True)
    words = done.numpy()
    for turn in (1, 2):
        got.token.fill_(-5)
        m.check(m.lib().ws_sample_batch_notify_host(torch.cuda.current_stream().cuda_stream, m.C.byref(got.desc), done.data_ptr(), turn), "ws_sample_batch_notify_host")
        until = time.monotonic() + 20.0
        while not (words == turn).all() and time.monotonic() < until:
            pass
        assert (words == turn).all(), words
        torch.cuda.synchronize()
        for k in ("token", "prob", "n_kept", "flags", "stats", "margin", "kept_ids", "kept_logits"):
            assert torch.equal(getattr(got, k), getattr(want, k)), k
    assert int(got.workspace.sum()) == 0 or not top_k and not min_p
    assert m.lib().ws_sample_batch_notify_host(None, m.C.byref(got.desc), None, 1) == -1


@pytest.mark.parametrize("vocab,n_hist,declared,flat,left", [(151936, 256, 256, False, False), (40003, 0, 0, False, False), (19471, 40, 12, False, True), (40003, 64, 64, True, True)])
def test_a_row_that_may_be_left(vocab, n_hist, declared, flat, left):
    """ws_sample_batch_try_host: the same answers, or - a row with more history than the batch declares, a row of equal logits, of which no list holds the top-k's
    ties - the mark in the flags and nothing else, the workspace zero; asked for again, the row is done as ever."""
    m = gc.pkg()
    rng = np.random.default_rng(vocab)
    x = torch.from_numpy((np.zeros((1, vocab)) if flat else rng.normal(0, 2, (1, vocab))).astype(np.float32)).cuda()
    args = dict(inv_t=np.full(1, 1.25, np.float32), top_p=np.full(1, 0.95), seed=np.full(1, 77 << 33, np.int64), step=np.full(1, 5, np.int64), top_k=np.full(1, 40, np.int32))
    hints = dict(top_k_max=40)
    if n_hist:
        args.update(hist=(rng.random(n_hist) ** 2 * vocab).astype(np.int32), hist_off=np.array([0, n_hist], np.int32), rep=np.full(1, 1.3, np.float32))
        hints.update(max_hist=declared)
    args = {k: pinned(v) for k, v in args.items()}
    make = lambda: m.BatchSampler(x, args["inv_t"], args["seed"], args["step"], kept_cap=64, **hints, **{k: v for k, v in args.items() if k not in ("inv_t", "seed", "step")})
    want, got = make().run(), make()
    got.token.fill_(-5)
    torch.cuda.synchronize()
    done = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    words = done.numpy()

    def ask(call, value):
        m.check(getattr(m.lib(), call)(torch.cuda.current_stream().cuda_stream, m.C.byref(got.desc), done.data_ptr(), value), call)
        until = time.monotonic() + 20.0
        while words[0] != value and time.monotonic() < until:
            pass
        assert words[0] == value
        torch.cuda.synchronize()

    ask("ws_sample_batch_try_host", 1)
    assert (int(got.flags[0]) == -1) == left
    assert int(got.workspace.sum()) == 0
    if left:
        assert int(got.token[0]) == -5
        ask("ws_sample_batch_notify_host", 2)
    for k in ("token", "prob", "n_kept", "flags", "stats", "margin", "kept_ids", "kept_logits"):
        assert torch.equal(getattr(got, k), getattr(want, k)), k
