"""DFA masks against the oracle's walk: state tables in LDS and past it, few
and many requested states (63 to 65 and more, repeats among them), sparse and
dense edges, vocabularies around a workgroup's 1024 tokens, tokens of no byte,
one byte and past 16 bytes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _vocabulary(rng, V):
    lengths = rng.choice([0, 1, 2, 5, 15, 16, 17, 40], V, p=[.1, .2, .2, .2, .1, .1, .05, .05])
    offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    return offsets, rng.integers(0, 256, int(offsets[-1]), dtype=np.uint8)


@pytest.mark.parametrize("n_states,density,V", [(96, 0.5, 5003), (96, 0.9, 5003), (97, 0.5, 5003), (97, 0.95, 5003),
                                                (96, 0.5, 200003), (8, 0.95, 200003)])
def test_masks_at_the_lines_between_the_kernels(oracle, n_states, density, V):
    """Requested states, table sizes, vocabularies and shares of surviving first bytes on both sides of
    every line that chooses the kernel; the vocabulary set after the DFA as well as before."""
    import gsample as gs

    rng = np.random.default_rng(V + n_states)
    offsets, data = _vocabulary(rng, V)
    nxt = np.where(rng.random((n_states, 256)) < density, rng.integers(0, n_states, (n_states, 256)), -1)
    nxt = nxt.astype(np.int32)
    finals = np.ones(n_states, np.uint8)
    viable = oracle.viable_states(nxt, finals)
    want = {q: oracle.dfa_legal_mask(nxt, viable, offsets, data, q) for q in range(min(n_states, 17))}
    s = gs.Sampler(vocab_size=V, max_rows=1)
    try:
        s.set_dfa(nxt, finals)
        s.set_vocab(offsets, data)
        for n in (1, 3, 4, 9, 10, 15, 16, 65):
            states = rng.integers(0, len(want), n)
            got = s.build_masks(states).cpu().numpy().view(np.uint32)
            for i, q in enumerate(states.tolist()):
                assert np.array_equal(got[i], want[q]), (n, i, q)
    finally:
        s.close()


@pytest.mark.parametrize("n_states,density", [(1, 0.9), (64, 0.1), (192, 0.5), (193, 0.995), (300, 0.1)])
@pytest.mark.parametrize("V", [1, 1023, 1025, 5003])
def test_masks_match_the_oracle(oracle, n_states, density, V):
    import gsample as gs

    rng = np.random.default_rng(V * 1000 + n_states)
    lengths = rng.choice([0, 1, 2, 5, 15, 16, 17, 40], V, p=[.1, .2, .2, .2, .1, .1, .05, .05])
    offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    data = rng.integers(0, 256, int(offsets[-1]), dtype=np.uint8)
    nxt = np.where(rng.random((n_states, 256)) < density, rng.integers(0, n_states, (n_states, 256)), -1)
    nxt = nxt.astype(np.int32)
    finals = (rng.random(n_states) < 0.5).astype(np.uint8)
    finals[0] = 1
    viable = oracle.viable_states(nxt, finals)
    s = gs.Sampler(vocab_size=V, max_rows=1)
    try:
        s.set_vocab(offsets, data)
        s.set_dfa(nxt, finals)
        for n in (1, 63, 64, 65, 130):
            states = rng.integers(0, n_states, n)
            got = s.build_masks(states).cpu().numpy().view(np.uint32)
            want = {int(q): oracle.dfa_legal_mask(nxt, viable, offsets, data, int(q)) for q in set(states.tolist())}
            for i, q in enumerate(states.tolist()):
                assert np.array_equal(got[i], want[q]), (n, i, q)
    finally:
        s.close()
