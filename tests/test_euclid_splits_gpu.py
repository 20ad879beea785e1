"""GPU parity of the per-stage Euclidean search with its codebook split over
many blocks (few tiles of frames, large codebooks: 8, 16 and 32 splits), at
the edges of the rule that picks the split, with repeated codes in different
splits; codes, distances and residual against the oracle, bit for bit."""

import numpy as np
import pytest

from test_euclid_gpu import bits, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,recipe,splits", [
    (3, 512, 1024, "higgs", 8),        # 128 codes a split
    (7, 768, 2048, "omnivoice", 16),
    (33, 768, 4096, "higgs", 32),
    (2, 512, 4096, "direct", 32),
    (4097, 512, 1024, "higgs", 4),     # 33 tiles: past the rule
])
def test_split_counts(monkeypatch, capfd, M, K, N, recipe, splits):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle

    print(f"[gpu] splits M={M} K={K} N={N} {recipe}", flush=True)
    monkeypatch.setenv("AQ_DEBUG", "1")
    cb = synth.normal(83, 1, (1, N, K))
    cb[0, N - 5] = cb[0, 5]   # equal codes, in the first and the last split
    x = synth.normal(83, 2, (M, K))
    x[0] = cb[0, 5]
    cfg = dict(x=x, M=M, K=K, Q=1, N=N, codebook=cb)
    out = run(torch, aqmi.Context(0), cb, getattr(aqmi, recipe.upper()), x)
    assert f"splits={splits},{splits}" in capfd.readouterr().err
    oracle = Oracle()
    ref = {"omnivoice": oracle.euclid_rvq, "higgs": oracle.higgs_rvq, "direct": oracle.direct_rvq}[recipe](cfg)
    dist = -ref["logit"] if recipe == "omnivoice" else ref["dist"]
    assert np.array_equal(out["idx"], ref["idx"])
    assert np.array_equal(bits(out["residual"]), bits(ref["residual"]))
    assert np.array_equal(bits(out["dist"]), bits(dist))


def test_refine_blocks_take_several_frames():
    """More open frames than the refine select launches blocks (16 per CU), at
    the width whose kernel holds the most: three codes 1e-3 apart share a lane's
    list of three keys in the sweep, which leaves their frames open, and fit its
    four in the split-fp16 pass, which settles them."""
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle

    M, K, N = 4600, 512, 1024
    print(f"[gpu] refine slots M={M} K={K} N={N}", flush=True)
    cb = synth.normal(87, 1, (N // 256, 4, 64, K))
    cb[:, 1:3] = cb[:, :1]   # codes 64 apart in a split are in one lane
    cb[:, 3] *= 1.5          # far from every frame
    cb = np.ascontiguousarray(cb.reshape(N, K) + synth.normal(87, 2, (N, K), 1e-3), np.float32)[None]
    x = synth.normal(87, 3, (M, K))
    out = run(torch, aqmi.Context(0), cb, aqmi.HIGGS, x)
    open_frames, scanned = int(out["fails"][0]), int(out["cbs"].exact_scans()[0])
    assert open_frames > 16 * torch.cuda.get_device_properties(0).multi_processor_count
    assert scanned < open_frames // 4   # the refine pass decided the rest
    ref = Oracle().higgs_rvq(dict(x=x, M=M, K=K, Q=1, N=N, codebook=cb))
    assert np.array_equal(out["idx"], ref["idx"])
    assert np.array_equal(bits(out["residual"]), bits(ref["residual"]))
    assert np.array_equal(bits(out["dist"]), bits(ref["dist"]))
