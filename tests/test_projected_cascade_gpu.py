"""GPU parity of the one-launch projected cascade (codebook width 64) at the
edges of its blocks: 4, 8 and 12 frames per block (AQ_PROJ_FRAMES asks for
them at any batch size), tails, F32 and Q8_0 weights and codebooks, hidden
sizes below the row stride, top-k, teacher forcing, codebooks of repeated
codes (whose tied frames the block scans exactly) and non-finite frames;
codes, residual and logits against the oracle, bit for bit."""

import numpy as np
import pytest

from test_euclid_gpu import bits, check_topk

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


@pytest.mark.parametrize("F", [4, 8, 12])
@pytest.mark.parametrize("M,recipe,H,N,cb_q8,proj_q8,topk,forced,special", [
    (2, 0, 256, 256, False, False, 0, False, ""),
    (11, 1, 1024, 1024, False, False, 4, False, ""),
    (13, 1, 512, 256, True, True, 0, True, ""),
    (25, 0, 1024, 512, False, True, 0, False, "nonfinite"),
    (40, 1, 768, 256, True, False, 2, False, "repeated"),
    (23, 0, 512, 256, False, False, 0, True, "repeated"),
])
def test_projected_cascade_block_edges(torch, ctx, oracle, monkeypatch, F, M, recipe, H, N, cb_q8, proj_q8, topk, forced,
                                       special):
    import aqmi
    from aqmi import synth

    print(f"[gpu] projected F={F} M={M} recipe={recipe} H={H} N={N} q8={cb_q8},{proj_q8} topk={topk} {special}", flush=True)
    monkeypatch.setenv("AQ_PROJ_FRAMES", str(F))
    Q = 3
    cfg = synth.projected_config(M, recipe, seed=71, H=H, N=N, Q=Q, cb_q8=cb_q8, proj_q8=proj_q8)
    cb = cfg["codebook_q8" if cb_q8 else "codebook"]
    if special == "repeated":
        for i in range(1, 8):   # more equal codes than keys kept per lane and wave
            cb[:, i * (N // 8):(i + 1) * (N // 8)] = cb[:, :N // 8]
    if special == "nonfinite":
        cfg["x"][1, 3] = np.inf
        cfg["x"][6, 100] = np.nan
        cfg["x"][9, 32:64] = synth.normal(71, 9, (32,), 1.0e-38)
    force = np.random.default_rng(5).integers(0, N, (M, Q)).astype(np.int32) if forced else None
    cbs = aqmi.Codebooks.projected(ctx, cb, cfg["w_in_q8" if proj_q8 else "w_in"], cfg["b_in"],
                                   cfg["w_out_q8" if proj_q8 else "w_out"], cfg["b_out"], recipe,
                                   aqmi.CB_Q8_0 if cb_q8 else aqmi.CB_F32, aqmi.CB_Q8_0 if proj_q8 else aqmi.CB_F32)
    x = torch.from_numpy(cfg["x"]).cuda()
    idx = torch.full((M, Q), -1, dtype=torch.int32, device="cuda")
    res = torch.empty((M, H), dtype=torch.float32, device="cuda")
    dist = torch.empty((M, Q), dtype=torch.float32, device="cuda")
    tki = torch.empty((M, Q, max(topk, 1)), dtype=torch.int32, device="cuda")
    tkd = torch.empty((M, Q, max(topk, 1)), dtype=torch.float32, device="cuda")
    cbs.encode(x, idx, res, dist, topk, tki if topk else None, tkd if topk else None,
               None if force is None else torch.from_numpy(force).cuda())
    torch.cuda.synchronize()
    if special == "repeated":
        assert cbs.exact_scans().sum() > 0   # tied frames took the block's exact scan
    ref = oracle.projected_rvq(cfg, force, topk=topk)
    got = dict(idx=idx.cpu().numpy(), residual=res.cpu().numpy(), dist=dist.cpu().numpy(), topk_idx=tki.cpu().numpy(),
               topk_dist=tkd.cpu().numpy())
    if special == "nonfinite":
        # x86's max keeps or drops a NaN by its place in the vector, so the
        # scale of a Q8_0 block with one is its own; the launches per stage
        # (fmaxf, every block alike) are this frame's reference
        monkeypatch.setenv("AQ_EUCLID_PIPELINE", "stages")
        cbs.encode(x, idx, res, dist, 0, None, None, None)
        torch.cuda.synchronize()
        for key, t in (("idx", idx), ("residual", res), ("dist", dist)):
            assert np.array_equal(got[key][6], t.cpu().numpy()[6], equal_nan=key != "idx")
            got[key][6] = ref[key][6]
    assert np.array_equal(got["idx"], ref["idx"])
    for key in ("residual", "dist"):
        a, b = got[key], ref[key]
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(bits(a[~np.isnan(a)]), bits(b[~np.isnan(b)]))
    if topk:
        check_topk(got, ref)


@pytest.mark.parametrize("F", [4, 8, 12])
@pytest.mark.parametrize("q8", [False, True])
def test_projected_cascade_channel_major(torch, ctx, oracle, monkeypatch, F, q8):
    """[B, C, T] input whose clips end inside the blocks (2 clips of 23 frames)."""
    import aqmi
    from aqmi import synth

    print(f"[gpu] projected channel-major F={F} q8={q8}", flush=True)
    monkeypatch.setenv("AQ_PROJ_FRAMES", str(F))
    B, T, H, N, Q = 2, 23, 1024, 256, 2
    cfg = synth.projected_config(B * T, aqmi.HIGGS, seed=73, H=H, N=N, Q=Q, cb_q8=q8, proj_q8=q8)
    cbt = aqmi.CB_Q8_0 if q8 else aqmi.CB_F32
    cb, w_in, w_out = (cfg[k + "_q8" if q8 else k] for k in ("codebook", "w_in", "w_out"))
    cbs = aqmi.Codebooks.projected(ctx, cb, w_in, cfg["b_in"], w_out, cfg["b_out"], aqmi.HIGGS, cbt, cbt)
    x = torch.from_numpy(np.ascontiguousarray(cfg["x"].reshape(B, T, H).transpose(0, 2, 1))).cuda()
    idx = torch.full((B * T, Q), -1, dtype=torch.int32, device="cuda")
    res = torch.empty((B * T, H), dtype=torch.float32, device="cuda")
    cbs.encode_strided(x, B * T, T, H * T, 1, T, idx, res)
    torch.cuda.synchronize()
    ref = oracle.projected_rvq(cfg)
    assert np.array_equal(idx.cpu().numpy(), ref["idx"])
    assert np.array_equal(bits(res.cpu().numpy()), bits(ref["residual"]))
