"""Typical-p over the whole vocabulary against the oracle: ids bit-exact, and
probabilities equal on replayed rows, within V 2^-52 relative of the oracle's
sequential sums on the rows that one pass settles. Sizes around the 16-byte
pieces and the workgroup's stride, rows at every alignment, equal logits in
one bin, heavy tails, softcap, and rows that only the replay settles."""
import ctypes as C

import numpy as np
import pytest

from oracle.oracle import Decoding

pytestmark = pytest.mark.gpu


def _rows(V, rng):
    n = rng.normal(0, 3, V)
    return {
        "normal": n,
        "grid": np.round(n * 4) / 4,
        "heavy": 8.0 * np.log((rng.permutation(V) + 1.0) ** -1.1) + rng.normal(0, 0.5, V),
        "narrow": 1.0 + 1e-3 * n,
        "equal": np.full(V, 1.5),
        "masked": np.where(rng.random(V) < 0.3, -np.inf, n),
    }


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V,pad", [(1023, 0), (1025, 3), (4097, 1), (16384, 8), (16391, 0), (70001, 2)])
def test_typical_rows_match_the_oracle(oracle, V, pad, dtype):
    import torch

    import gsample as gs

    rng = np.random.default_rng(V)
    xs, cfgs, us, caps, names = [], [], [], [], []
    for name, x in _rows(V, rng).items():
        for p in (0.02, 0.5, 0.9, 0.999):
            for T in (0.3, 1.0):
                xs.append(x)
                names.append(name)
                caps.append(20.0 if p == 0.5 else 0.0)
                us.append(float(rng.random()))
                cfgs.append(gs.DecodingConfig(temperature=T, topK=0, topP=1.0, typicalP=p, repetitionPenalty=1.0,
                                              repetitionWindow=0))
    wide = np.zeros((len(xs), V + pad), np.float32)
    wide[:, :V] = np.stack(xs)
    logits = torch.from_numpy(wide).to(torch.float32 if dtype == "f32" else torch.bfloat16)
    values = logits.to(torch.float32).numpy()[:, :V]
    s = gs.Sampler(vocab_size=V, max_rows=len(xs))
    try:
        conf = np.stack([gs.runtime.row_config(c, uniform=u, softcap_value=k) for c, u, k in zip(cfgs, us, caps)])
        out = s.sample(logits.cuda()[:, :V], conf)
    finally:
        s.close()
    settled = 0
    for r, c in enumerate(cfgs):
        x = oracle.softcap(values[r], caps[r]) if caps[r] > 0 else values[r]
        t, tr = oracle.sample_token(x, [], Decoding(temperature=c.temperature, topK=0, topP=1.0, minP=0.0,
                                                    typicalP=c.typicalP, repetitionPenalty=1.0,
                                                    repetitionWindow=0), us[r])
        assert int(out.tokens[r]) == t, (names[r], c.typicalP, c.temperature, int(out.tokens[r]), t)
        if out.flags[r] & gs.GS_FLAG_EXACT_PATH:
            assert out.probabilities[r] == tr.probability, (names[r], r)
            assert names[r] != "normal" or c.typicalP > 0.99 or V < 4096, (names[r], r)
        else:
            settled += 1
            # (the softcap makes -inf finite)
            assert names[r] != "equal" and (names[r] != "masked" or caps[r] > 0), (names[r], r)
            assert abs(out.probabilities[r] - tr.probability) <= V * 2.0 ** -52 * tr.probability, (names[r], r)
    assert settled >= len(cfgs) // 3, settled


def _softmax(x, T):
    """Probabilities and surprises of a row in binary64 (the typical order's inputs)."""
    v = x.astype(np.float64) / T
    p = np.exp(v - v.max())
    p /= p.sum()
    return p, np.abs(-np.log(p) + np.sum(p * np.log(p)))


def _cuts_within(x, T, group, fractions, picks):
    """(typicalP, u) with the typical cut inside the items `group` (a boolean mask of equal surprise), at the
    fractions of their mass (never at an item's end), and draws at the picks of the kept part of it."""
    p, s = _softmax(x, T)
    edge = s[group].max() + 1e-9
    nearer = (s < edge) & ~group
    before, mass = p[nearer].sum(), p[group].sum()
    above = p[nearer & (p > p[group].max())].sum()
    n = int(group.sum())
    for f in fractions:
        f = (np.floor(f * n) + 0.4) / n
        kept = before + f * mass
        for g in picks:
            yield kept, (above + g * f * mass) / kept


def _check_rows(oracle, rows, dtype):
    """Samples rows [(name, x, T, typicalP, u)]; ids must be the oracle's. Returns which were replayed."""
    import torch

    import gsample as gs

    V = len(rows[0][1])
    x = torch.from_numpy(np.stack([r[1] for r in rows]).astype(np.float32)).to(dtype)
    cfgs = [gs.DecodingConfig(temperature=r[2], topK=0, topP=1.0, typicalP=r[3], repetitionPenalty=1.0,
                              repetitionWindow=0) for r in rows]
    s = gs.Sampler(vocab_size=V, max_rows=len(rows))
    try:
        conf = np.stack([gs.runtime.row_config(c, uniform=r[4]) for c, r in zip(cfgs, rows)])
        out = s.sample(x.cuda(), conf)
    finally:
        s.close()
    values = x.to(torch.float32).numpy()
    for i, (name, _, T, p, u) in enumerate(rows):
        t, _ = oracle.sample_token(values[i], [], Decoding(temperature=T, topK=0, topP=1.0, minP=0.0, typicalP=p,
                                                           repetitionPenalty=1.0, repetitionWindow=0), u)
        assert int(out.tokens[i]) == t, (name, T, p, u, int(out.tokens[i]), t)
    return (out.flags & gs.GS_FLAG_EXACT_PATH) != 0


def _zeros_rows(rng, V=2048):
    """Rows of a grid with zeros of both signs mixed, the cut and the draw among the zeros."""
    for step in (0.25, 0.125, 0.5):
        x = np.round(rng.normal(0, 3, V) / step) * step
        x[rng.random(V) < 0.15] = 0.0
        x = np.where((x == 0) & (rng.random(V) < 0.5), -0.0, x)
        for T in (0.7, 1.3):
            for p, u in _cuts_within(x, T, x == 0, (0.2, 0.5, 0.8), (0.1, 0.5, 0.9)):
                yield f"zeros {step}", x, T, p, u


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_typical_cut_among_signed_zeros(oracle, dtype):
    """+0 and -0 are equal: the zeros kept are the ones of the lowest ids, whatever their sign."""
    import torch

    rows = list(_zeros_rows(np.random.default_rng(5)))
    replayed = _check_rows(oracle, rows, getattr(torch, dtype))
    assert not replayed.any(), np.nonzero(replayed)[0]


def _mirrored_rows(rng, V=2048):
    """Two groups of equal logits on either side of the mean, their surprises equal to rounding (the temperature
    is found by bisection: 2 E[l] = 7 + 5), the cut among them."""
    x = np.round(rng.normal(0, 3, V) * 8) / 8
    x[(x == 7) | (x == 5)] = 0.125
    ids = rng.permutation(V)
    x[ids[:40]], x[ids[40:100]] = 7.0, 5.0
    lo, hi = 0.3, 6.0  # E[l] falls as the temperature rises
    for _ in range(200):
        T = 0.5 * (lo + hi)
        lo, hi = (T, hi) if float(np.sum(_softmax(x, T)[0] * x)) > 6.0 else (lo, T)
    group = (x == 7) | (x == 5)
    for T in (lo, hi, lo * (1 - 4e-16), hi * (1 + 4e-16), lo * (1 + 4e-15)):
        for p, _ in _cuts_within(x, T, group, (0.2, 0.5, 0.8), (0.5,)):
            for u in rng.random(6):
                yield "mirrored", x, T, p, float(u)


def _tiny_rows(rng, V=2048):
    """Zeros with a few 3e-17 among them: other logits of the same surprise, the cut and the draw in the zeros."""
    x = np.round(rng.normal(0, 3, V) * 4) / 4
    x[rng.random(V) < 0.15] = 0.0
    zeros = np.nonzero(x == 0)[0]
    group = x == 0
    x[zeros[[1, len(zeros) // 2, -1]]] = 3e-17
    for T in (0.7, 1.3):
        for p, u in _cuts_within(x, T, group, (0.2, 0.5, 0.8), (0.1, 0.5, 0.9)):
            yield "tiny", x, T, p, u


@pytest.mark.parametrize("make", [_mirrored_rows, _tiny_rows])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_typical_cut_between_equal_surprises(oracle, dtype, make):
    """Different logits of one surprise at the cut: the reference's rounding orders them, however many
    equal logits lie between the cut and the next different one, so the replay decides."""
    import torch

    assert _check_rows(oracle, list(make(np.random.default_rng(5))), getattr(torch, dtype)).all()


def _drawn(x, T):
    """(typicalP, u) of draws in the middle of a row's zeros, the cut elsewhere."""
    p, _ = _softmax(x, T)
    zero = np.abs(x) < 1e-9
    above, mass = p[x > 0.1].sum(), p[zero].sum()
    return [(0.9999, (above + g * mass) / 0.9999) for g in (0.3, 0.5, 0.7)]


def _tiny_drawn_rows(rng, V=2048):
    """Zeros with a few 3e-17 among them, and zeros that start a bin (the row spans 64 grid steps, a power of
    two) with a few 2e-15 at the end of the bin above."""
    x = next(_tiny_rows(rng, V))[1]
    for T in (1.3, 2.0):
        for p, u in _drawn(x, T):
            yield "tiny drawn", x, T, p, u
    for _, x, T, p, u in list(_bin_edge_rows(rng, V)):
        x = x.copy()
        x[np.nonzero(x == 0)[0][[3, -2]]] = 2e-15
        yield "tiny above the bin", x, T, p, u


def _bin_edge_rows(rng, V=2048):
    x = np.clip(np.round(rng.normal(0, 3, V) * 4) / 4, -8, 8)
    x[[17, 1900]] = 8.0, -8.0
    for p, u in _drawn(x, 1.0):
        yield "bin edge", x, 1.0, p, u


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_typical_draw_between_equal_probabilities(oracle, dtype):
    """Different logits whose probabilities could round out of order around the drawn one: the replay decides,
    also with equal logits between them and the drawn one, or a bin's edge. A run of equal logits
    at a bin's edge with nothing beyond it is settled."""
    import torch

    assert _check_rows(oracle, list(_tiny_drawn_rows(np.random.default_rng(5))), getattr(torch, dtype)).all()
    assert not _check_rows(oracle, list(_bin_edge_rows(np.random.default_rng(5))), getattr(torch, dtype)).any()


@pytest.mark.parametrize("V", [17, 40, 64, 65])
def test_typical_rows_are_decided_once(oracle, V):
    """A topK of the whole vocabulary: up to 64 the finish settles such rows (its flags and probabilities
    stay, with the batch's typical-p hint too), past it the typical-p kernel. Through a context and
    through the entry point with two replay slots."""
    import torch

    import gsample as gs

    rng = np.random.default_rng(V)
    rows, R = [], 48
    for i in range(R):
        x = np.full(V, 1.5) if i % 4 == 3 else rng.normal(0, 3, V)
        rows.append(np.round(x * 4) / 4 if i % 2 else x)
    x = torch.from_numpy(np.stack(rows).astype(np.float32)).cuda()
    us = rng.random(R)
    cfgs = [gs.DecodingConfig(temperature=0.8, topK=max(V, 64) if i % 3 == 0 else V, topP=1.0,
                              typicalP=float(rng.uniform(0.2, 0.99)), repetitionPenalty=1.0, repetitionWindow=0)
            for i in range(R)]
    conf = np.stack([gs.runtime.row_config(c, uniform=u) for c, u in zip(cfgs, us)])
    s = gs.Sampler(vocab_size=V, max_rows=R)
    try:
        plain = s.sample(x, conf, hints=0)
        out = s.sample(x, conf)
        assert s.prepare(x, conf)[0].hints & gs.runtime.GS_BATCH_TYPICAL
        b, keep = s.prepare(x, conf)
        res = torch.zeros((R, 2), dtype=torch.float64, device="cuda")
        b.results = res.data_ptr()
        torch.cuda.synchronize()
        stream = torch.cuda.Stream()
        assert gs.runtime.library().gs_sample_noalloc(C.byref(b), V, C.c_void_p(stream.cuda_stream)) == 0
        stream.synchronize()
        fixed = res.cpu().numpy().view(np.uint8).reshape(-1).view(gs.runtime.RESULT_DTYPE)
    finally:
        s.close()
    for i, c in enumerate(cfgs):
        t, _ = oracle.sample_token(x[i].cpu().numpy(), [], Decoding(
            temperature=c.temperature, topK=c.topK, topP=1.0, minP=0.0, typicalP=c.typicalP, repetitionPenalty=1.0,
            repetitionWindow=0), us[i])
        assert int(plain.tokens[i]) == int(out.tokens[i]) == int(fixed["token"][i]) == t, i
    assert np.array_equal(out.flags, fixed["flags"])
    assert np.array_equal(out.probabilities, fixed["probability"])
    if V <= 64:
        assert np.array_equal(out.flags, plain.flags) and np.array_equal(out.probabilities, plain.probabilities)
    else:
        assert (plain.flags & gs.GS_FLAG_EXACT_PATH).all() and not (out.flags & gs.GS_FLAG_EXACT_PATH).all()


def test_typical_launch_is_timed():
    """The typical-p kernel's time is in the deep stage, alone and after full-vocabulary draws."""
    import torch

    import gsample as gs

    V = 50000
    x = torch.from_numpy(np.random.default_rng(3).normal(0, 3, (8, V)).astype(np.float32)).cuda()
    draw = gs.DecodingConfig(temperature=0.8, topK=0, topP=1.0, typicalP=1.0, repetitionPenalty=1.0, repetitionWindow=0)
    s = gs.Sampler(vocab_size=V, max_rows=8)
    try:
        for n in (0, 4, 8):  # typical-p rows among full-vocabulary draws
            conf = np.stack([gs.runtime.row_config(draw.merged(typicalP=0.9 if i < n else 1.0), uniform=0.3)
                             for i in range(8)])
            b, keep = s.prepare(x, conf)
            want = (gs.runtime.GS_BATCH_TYPICAL if n else 0) | (gs.runtime.GS_BATCH_FULL_DRAWS if n < 8 else 0)
            assert b.hints == want
            s.launch(b)
            s.synchronize()
            s.timing_begin(3)
            for _ in range(3):
                s.launch(b)
            ms, calls = s.timing_end()["deep"]
            assert calls == 3 and ms > 3 * (0.03 if n else 0.0), (n, ms, calls)
    finally:
        s.close()
