"""GPU parity of the per-stage Euclidean search with its codebook split over
many blocks (few tiles of frames, large codebooks: 8, 16 and 32 splits), at
the edges of the rule that picks the split, with repeated codes in different
splits; codes, distances and residual against the oracle, bit for bit."""

import numpy as np
import pytest

from test_euclid_gpu import bits, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,recipe", [
    (3, 512, 1024, "higgs"),        # 8 splits of 128 codes
    (7, 768, 2048, "omnivoice"),    # 16
    (33, 768, 4096, "higgs"),       # 32
    (2, 512, 4096, "direct"),       # 32
    (4097, 512, 1024, "higgs"),     # 33 tiles: past the rule, 4
])
def test_split_counts(M, K, N, recipe):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle

    print(f"[gpu] splits M={M} K={K} N={N} {recipe}", flush=True)
    cb = synth.normal(83, 1, (1, N, K))
    cb[0, N - 5] = cb[0, 5]   # equal codes, in the first and the last split
    x = synth.normal(83, 2, (M, K))
    x[0] = cb[0, 5]
    cfg = dict(x=x, M=M, K=K, Q=1, N=N, codebook=cb)
    out = run(torch, aqmi.Context(0), cb, getattr(aqmi, recipe.upper()), x)
    oracle = Oracle()
    ref = {"omnivoice": oracle.euclid_rvq, "higgs": oracle.higgs_rvq, "direct": oracle.direct_rvq}[recipe](cfg)
    dist = -ref["logit"] if recipe == "omnivoice" else ref["dist"]
    assert np.array_equal(out["idx"], ref["idx"])
    assert np.array_equal(bits(out["residual"]), bits(ref["residual"]))
    assert np.array_equal(bits(out["dist"]), bits(dist))
