"""GPU parity of the narrow Euclidean cascade (K = 256) at the edges of its
tiles: one, two and four frame groups per block (AQ_EUCLID_PIPELINE=narrow1,
narrow2, narrow4 ask for them at any batch size), frame counts around whole
groups and blocks, codebooks that give some of the eight waves no or one
16-code block, every recipe, top-k and teacher forcing; codes, residuals,
distances and top-k against the oracle, bit for bit."""

import numpy as np
import pytest

from test_euclid_gpu import bits, check_topk, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t

    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.fixture(scope="module")
def ctx(torch):
    import aqmi

    return aqmi.Context(0)


@pytest.fixture(scope="module")
def oracle():
    from oracle import Oracle

    return Oracle()


def reference_topk(oracle, recipe, cfg, ref, force, topk):
    """The topk best codes per frame and stage from every code's value, each
    computed by the oracle as a codebook of that one code (four times over,
    which keeps the summation order)."""
    r = np.ascontiguousarray(cfg["x"], np.float32).copy()
    idx, logit = [], []
    for s in range(cfg["Q"]):
        book = cfg["codebook"][s]
        value = np.empty((cfg["M"], cfg["N"]), np.float32)
        for n in range(cfg["N"]):
            one = dict(x=r, M=cfg["M"], K=cfg["K"], Q=1, N=4, codebook=np.repeat(book[n:n + 1], 4, 0)[None])
            value[:, n] = (oracle.euclid_rvq(one)["logit"] if recipe == "omnivoice" else -oracle.direct_rvq(one)["dist"])[:, 0]
        order = np.argsort(-value.astype(np.float64), axis=1, kind="stable")[:, :topk]
        idx.append(order.astype(np.int32))
        logit.append(np.take_along_axis(value, order, 1))
        r = r - book[(ref["idx"] if force is None else force)[:, s]]
    return dict(topk_idx=np.stack(idx, 1), topk_logit=np.stack(logit, 1))


@pytest.mark.parametrize("fg", [1, 2, 4])
@pytest.mark.parametrize("M,N,recipe,q8,topk,forced", [
    (1, 64, "omnivoice", False, 0, False),      # one frame (vec_dot order), four waves without codes
    (15, 64, "direct", False, 4, False),
    (16, 192, "higgs", False, 1, True),         # waves 4 .. 7 with one block
    (17, 192, "omnivoice", False, 0, True),
    (63, 1088, "direct", False, 0, False),      # an odd number of blocks per wave
    (64, 2048, "higgs", True, 4, False),
    (65, 1088, "higgs", True, 0, True),
    (129, 2048, "omnivoice", False, 3, False),
])
def test_narrow_cascade_tile_edges(torch, ctx, oracle, monkeypatch, fg, M, N, recipe, q8, topk, forced):
    import aqmi
    from aqmi import synth

    print(f"[gpu] narrow fg={fg} M={M} N={N} {recipe} q8={q8} topk={topk} forced={forced}", flush=True)
    monkeypatch.setenv("AQ_EUCLID_PIPELINE", f"narrow{fg}")
    Q, K = 3, 256
    x = synth.normal(61, 1, (M, K))
    cfg = dict(x=x, M=M, K=K, Q=Q, N=N)
    if q8:
        cb = cfg["codebook_q8"] = np.stack([synth.q8_0_random_codebook(61, 10 + 10 * s, N, K) for s in range(Q)])
    else:
        cb = cfg["codebook"] = np.stack([synth.normal(61, 10 + 10 * s, (N, K), 1.0 / 16.0) for s in range(Q)])
    force = np.random.default_rng(5).integers(0, N, (M, Q)).astype(np.int32) if forced else None
    out = run(torch, ctx, cb, getattr(aqmi, recipe.upper()), x, cb_type=aqmi.CB_Q8_0 if q8 else aqmi.CB_F32,
              topk=topk, force=force)
    if recipe == "omnivoice":
        ref = oracle.euclid_rvq(cfg, force)
        dist = -ref["logit"]
    elif recipe == "higgs":
        ref = oracle.higgs_rvq(cfg, force, topk=topk)
        dist = ref["dist"]
    else:
        ref = oracle.direct_rvq(cfg, force)
        dist = ref["dist"]
    assert np.array_equal(out["idx"], ref["idx"])
    assert np.array_equal(bits(out["residual"]), bits(ref["residual"]))
    assert np.array_equal(bits(out["dist"]), bits(dist))
    if topk:
        if "topk_idx" not in ref:
            ref.update(reference_topk(oracle, recipe, cfg, ref, force, topk))
        check_topk(out, ref)
