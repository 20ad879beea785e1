"""The images that an upload builds for the one-launch cascades alone: an
upload without memory for them, or for what comes after them, is not refused
and its calls give the same bits through the per-stage launches
(AQ_EUCLID_TEST_NO_IMAGE ends the memory),
and shapes that those cascades do not take hold none."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t

    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def encode(torch, cbs, x, want_launches):
    M = x.shape[0]
    idx = torch.full((M, cbs.Q), -1, dtype=torch.int32, device="cuda")
    res = torch.empty((M, cbs.H), dtype=torch.float32, device="cuda")
    cbs.ctx.set_timing(True)
    cbs.encode(x, idx, res)
    assert len(cbs.ctx.read_timing()) == want_launches   # one per stage, or one for all
    cbs.ctx.set_timing(False)
    return idx.cpu().numpy(), res.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("kind,ends", [
    ("plain", "at"), ("plain", "after"), ("q8", "at"), ("ema", "at"), ("ema", "after"), ("projected", "at"),
    ("projected_q8", "at")])
def test_upload_without_memory_for_images(torch, monkeypatch, kind, ends):
    import aqmi
    from aqmi import synth

    print(f"[gpu] upload images {kind} {ends}", flush=True)
    ctx, Q, M = aqmi.Context(0), 3, 70

    def upload():
        if kind == "plain":
            return aqmi.Codebooks(ctx, synth.normal(95, 1, (Q, 256, 256)), aqmi.OMNIVOICE)
        if kind == "q8":
            blocks = np.stack([synth.q8_0_random_codebook(95, 10 + s, 256, 256) for s in range(Q)])
            return aqmi.Codebooks(ctx, blocks, aqmi.HIGGS, aqmi.CB_Q8_0)
        if kind == "ema":
            return aqmi.Codebooks.from_ema(ctx, synth.normal(95, 1, (Q, 256, 256)), np.ones((Q, 256), np.float32),
                                           aqmi.DIRECT)
        q8 = kind == "projected_q8"
        cfg = synth.projected_config(M, aqmi.HIGGS, seed=95, H=512, N=256, Q=Q, proj_q8=q8)
        return aqmi.Codebooks.projected(ctx, cfg["codebook"], cfg["w_in_q8" if q8 else "w_in"], cfg["b_in"],
                                        cfg["w_out_q8" if q8 else "w_out"], cfg["b_out"], aqmi.HIGGS, aqmi.CB_F32,
                                        aqmi.CB_Q8_0 if q8 else aqmi.CB_F32)

    cbs = upload()
    x = torch.from_numpy(synth.normal(95, 2, (M, cbs.H))).cuda()
    want = encode(torch, cbs, x, 1)
    monkeypatch.setenv("AQ_EUCLID_TEST_NO_IMAGE", ends)
    got = encode(torch, upload(), x, Q)
    assert np.array_equal(got[0], want[0])
    assert np.array_equal(got[1], want[1])


def test_no_image_where_no_call_reads_it(torch):
    """4 096 codes are past the projected cascade's 2 048: 64 stages would hold
    48 MiB of images."""
    import aqmi
    from aqmi import synth

    print("[gpu] upload images past the shapes", flush=True)
    ctx, Q, N, K, H = aqmi.Context(0), 64, 4096, 64, 1024
    cb, w = synth.normal(96, 1, (Q, N, K)), synth.normal(96, 2, (Q, K, H))
    one = aqmi.Codebooks.projected(ctx, cb[:1], w[:1], None, np.ascontiguousarray(w[:1].transpose(0, 2, 1)), None, aqmi.HIGGS)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    cbs = aqmi.Codebooks.projected(ctx, cb, w, None, np.ascontiguousarray(w.transpose(0, 2, 1)), None, aqmi.HIGGS)
    held = before - torch.cuda.mem_get_info()[0]
    # fp32 codes and two fp16 images, the project_out table, both projections,
    # three values per code
    need = Q * (N * K * 8 + N * H * 4 + 2 * K * H * 4 + N * 12)
    print(f"held {held}, needed {need}", flush=True)
    # the three 1 MiB buffers of values per code can lie in a chunk that the
    # process holds already; the others are 16 MiB at least
    assert held >= need - 3 * Q * N * 4 - (2 << 20)
    assert held < need + (32 << 20)   # the allocator's rounding of ten buffers
    del one, cbs
