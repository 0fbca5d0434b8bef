"""GPU: the walk over a sequence's verify positions (ws_accept_sampled, ws_accept_sampled_fresh, ws_history_stage) against the rules written out position
by position (src/sampling/acceptor.cpp:63-100, include/whirl/relax_accept.h:72-96): every number of drafts, rows without a usable token, typical
drafts, entropies near their threshold, texts that repeat, slots without room. Whole numbers, so exactly."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

import gpu_cases as gc

EPS, DELTA, HOST, NEAR, FULL = 0.09, 0.3, 1, 2, 4
ALL_MASKED, APPROX = 8, 128


def extends_repeat(text, n=6, window=4096):
    """text: history and tail; the window counts the history's part alone, which the callers here keep below it."""
    last = text[-n:]
    return len(text) >= n + 1 and any(text[i:i + n] == last for i in range(len(text) - n))


def walk(tok, fl, nd, drafts, typical, pd, ent, text, nxt, cap):
    """One sequence: (accepted, chosen, status, relaxed, kept words or None)."""
    if text is not None and len(text) + 2 + nd > cap:
        return 0, -1, FULL | HOST, 0, {}
    acc, st, relaxed, words = 0, 0, 0, {}
    while True:
        if tok[acc] < 0 or fl[acc] & ALL_MASKED:
            st |= HOST
            break
        if typical and acc < nd:
            thr = min(float(np.float32(EPS)), float(np.float32(DELTA)) * math.exp(-ent[acc]))
            if fl[acc] & APPROX and abs(pd[acc] - thr) < 0.02 * thr:
                st |= NEAR
            if pd[acc] >= thr and not (text is not None and extends_repeat(text + [nxt] + drafts[:acc + 1])):
                words[acc] = drafts[acc]
                acc, relaxed = acc + 1, relaxed + 1
                continue
        words[acc] = int(tok[acc])
        if acc == nd or tok[acc] != drafts[acc]:
            break
        acc += 1
    return acc, int(tok[acc]), st, relaxed, words


@pytest.mark.gpu
@pytest.mark.parametrize("fresh", [True, False])
@pytest.mark.parametrize("typical,history", [(False, False), (True, False), (False, True), (True, True)])
def test_walk(typical, history, fresh):
    m = gc.pkg()
    rng = np.random.default_rng(5 + 2 * typical + history)
    n_seq, cap = 97, 64
    nd = np.array([i % 16 for i in range(n_seq)])
    row0 = np.cumsum([0] + list(nd + 1))[:-1]
    rows = int((nd + 1).sum())
    drafts = [list(map(int, rng.integers(0, 3, k))) for k in nd]  # (three tokens: texts repeat)
    tok = rng.integers(0, 3, rows).astype(np.int32)
    for s in range(n_seq):  # most drafts are what was drawn
        for j in range(nd[s]):
            if rng.random() < 0.85:
                tok[row0[s] + j] = drafts[s][j]
    tok[rng.random(rows) < 0.02] = -1
    fl = np.where(rng.random(rows) < 0.02, ALL_MASKED, 0) | np.where(rng.random(rows) < 0.5, APPROX, 0)
    ent = rng.uniform(0.0, 3.0, rows)
    thr = np.minimum(np.float64(np.float32(EPS)), np.float64(np.float32(DELTA)) * np.exp(-ent))
    pd = thr * rng.choice([0.5, 0.985, 1.015, 2.0], rows)
    text = [list(map(int, rng.integers(0, 3, rng.integers(0, cap - 1)))) for _ in range(n_seq)]
    nxt = rng.integers(0, 3, n_seq)
    ctl = torch.full((n_seq, m.CTL_WORDS), -7, dtype=torch.int32)
    for s in range(n_seq):
        ctl[s, 16:16 + nd[s]] = torch.tensor(drafts[s], dtype=torch.int32)
        ctl[s, 48] = int(nd[s])
    before = ctl.clone()
    dev = "cuda:0"
    ctl = ctl.to(dev)
    t = lambda a, dt=None: torch.as_tensor(np.ascontiguousarray(a), dtype=dt).to(dev)
    area, r0 = t(np.arange(n_seq) * m.CTL_WORDS, torch.int32), t(row0, torch.int32)
    H, slot = m.DeviceHistory(n_seq, cap, dev), t(rng.permutation(n_seq), torch.int32)
    place = slot.cpu().numpy()
    for s in range(n_seq):
        H.tokens[place[s], :len(text[s])] = t(text[s], torch.int32)
        H.tokens[place[s], len(text[s])] = int(nxt[s])
        H.len[place[s]] = len(text[s])
    H.n_gen.copy_(torch.arange(n_seq, dtype=torch.int64))
    if history:
        out = {k: torch.full((rows,), -9, dtype=torch.int32, device=dev) for k in ("off", "len", "query")}
        step = torch.full((rows,), -9, dtype=torch.int64, device=dev)
        status = m.history_stage(H, slot, ctl, area, r0, out["off"], out["len"], out["query"], step).cpu().numpy()
        for s in range(n_seq):
            room = len(text[s]) + 2 + nd[s] <= cap
            at = slice(int(row0[s]), int(row0[s] + nd[s] + 1))
            j = np.arange(nd[s] + 1)
            assert status[s] == (0 if room else FULL), s
            assert (out["off"][at].cpu().numpy() == place[s] * cap).all() and (step[at].cpu().numpy() == place[s] + j).all(), s
            assert (out["len"][at].cpu().numpy() == (len(text[s]) + 1 + j if room else 0)).all(), s
            assert out["query"][at].tolist() == drafts[s] + [-1], s
    i32 = lambda v: torch.full((n_seq,), v, dtype=torch.int32, device=dev)
    n_acc, chosen, st, relaxed = i32(-5), i32(-5), i32(-5), i32(40)
    keep = (t(tok), t(fl, torch.int32), t(pd, torch.float64), t(ent, torch.float64))
    a = m.Accept(token=keep[0].data_ptr(), flags=keep[1].data_ptr(), row0=r0.data_ptr(), ctl_all=ctl.data_ptr(), area=area.data_ptr(), n_seq=n_seq,
                 n_accepted=n_acc.data_ptr(), chosen=chosen.data_ptr(), status=st.data_ptr(), typical=int(typical), query_prob=keep[2].data_ptr(),
                 entropy=keep[3].data_ptr(), eps=EPS, delta=DELTA, relaxed=relaxed.data_ptr())
    if history:
        a.hist = H.ref(slot)
    fn = m.lib().ws_accept_sampled_fresh if fresh else m.lib().ws_accept_sampled
    assert fn(torch.cuda.current_stream().cuda_stream, C.byref(a)) == 0
    after, tokens = ctl.cpu(), H.tokens.cpu().numpy()
    seen = set()
    for s in range(n_seq):
        at = slice(int(row0[s]), int(row0[s] + nd[s] + 1))
        w = walk(tok[at], fl[at], int(nd[s]), drafts[s], typical, pd[at], ent[at], text[s] if history else None, int(nxt[s]), cap)
        got = int(n_acc[s]), int(chosen[s]), int(st[s]), int(relaxed[s]) - (0 if fresh or w[2] & FULL else 40)
        assert got == w[:4] or (not fresh and w[2] & FULL and got == w[:3] + (40,)), (s, got, w)
        want = before[s].clone()
        for j, v in w[4].items():
            want[j] = v
        assert torch.equal(after[s], want), s
        if history:
            ok = not w[2] & HOST
            full = text[s] + [int(nxt[s])] + drafts[s][:w[0]] + [w[1]] if ok else text[s] + [int(nxt[s])]
            assert tokens[place[s]][:len(full)].tolist() == full and int(H.len[place[s]]) == len(full) - 1, s
            assert int(H.n_gen[place[s]]) == place[s] + (w[0] + 1 if ok else 0), s
        seen |= {w[2], ("acc", w[0] > 4), ("relaxed", w[3] > 0)}
    assert HOST in seen and ("acc", True) in seen and (not typical or ("relaxed", True) in seen) and (not history or FULL | HOST in seen)
