"""tokenLogProbability (sampling.ts:67-80) over row lengths, row strides that
leave rows off the 16-byte grid, both element types, and rows whose maximum is
not finite, against numpy in binary64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one element, less than a 16-byte piece, around a thread's and a part's share,
# odd and whole multiples; row counts on both sides of one part per row
@pytest.mark.parametrize("vocab,rows", [(1, 3), (3, 2), (7, 5), (1023, 4), (4096, 5), (8192, 3), (8193, 33), (40001, 3), (262144, 2),
                                        (151643, 1), (4099, 2100)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_log_prob_rows(vocab, rows, dtype):
    import torch

    import gsample as gs

    rng = np.random.default_rng(vocab + rows)
    pad = 3  # an odd stride: rows start at every alignment an element allows
    x = torch.from_numpy(rng.normal(0, 4, (rows, vocab + pad)).astype(np.float32))
    x = x if dtype == "f32" else x.to(torch.bfloat16)
    x[:, vocab:] = float("nan")  # never read
    if vocab > 2 and rows > 2:
        x[0, : vocab // 2] = -float("inf")
        x[1, 1] = float("nan")
        x[2, 2] = float("inf")
    if rows > 3:
        x[3, :vocab] = -float("inf")
    toks = rng.integers(0, vocab, rows).astype(np.int32)
    if rows > 4:
        toks[4] = vocab
    s = gs.Sampler(vocab_size=vocab, max_rows=1)
    try:
        got = s.token_log_probability(x.cuda(), toks)
    finally:
        s.close()
    v = x[:, :vocab].to(torch.float64).numpy()
    for r in range(rows):
        with np.errstate(all="ignore"):
            m = v[r].max()
            want = v[r, toks[r]] - m - np.log(np.exp(v[r] - m).sum()) if toks[r] < vocab else np.nan
        if np.isfinite(want):
            # the sum's relative error: a thread adds at most V / 256 terms of
            # one ulp each one after another when the row is one part, and the
            # joins add a few more; then the result's own roundings
            bound = (vocab / 256 + 40) * 2.0 ** -52 + 4 * np.spacing(abs(want) + abs(m))
            assert abs(got[r] - want) <= bound, (r, got[r], want)
        else:
            assert np.array_equal(got[r], want, equal_nan=True), (r, got[r], want)
