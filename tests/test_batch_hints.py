"""The hints a batch carries follow its rows' options, whatever their number."""
import itertools

import numpy as np


def test_batch_hints():
    import gsample as gs
    from gsample import runtime as rt

    V = 100
    rows = []
    for t, k, p, m, ty, mask in itertools.product((0.0, 0.7), (0, 40, V, V + 1), (0.9, 1.0), (0.0, 0.1), (0.9, 1.0),
                                                  (-1, 0)):
        c = gs.DecodingConfig(temperature=t, topK=k, topP=p, minP=m, typicalP=ty)
        free = t > 0 and p >= 1 and m == 0 and mask < 0
        want = (rt.GS_BATCH_FULL_DRAWS if free and ty >= 1 and k == 0 else 0)
        want |= rt.GS_BATCH_TYPICAL if free and ty < 1 and (k == 0 or k >= V) else 0
        conf = np.stack([rt.row_config(c, uniform=0.5, mask_slot=mask)])
        assert rt.batch_hints(conf, V) == want
        assert bool(want & rt.GS_BATCH_FULL_DRAWS) == rt.full_draw_rows(conf)
        rows.append((conf, want))
    rng = np.random.default_rng(1)
    for _ in range(50):
        pick = [rows[i] for i in rng.integers(0, len(rows), int(rng.integers(2, 5)))]
        want = 0
        for _, w in pick:
            want |= w
        assert rt.batch_hints(np.concatenate([c for c, _ in pick]), V) == want
