"""GPU parity of the DAC cascade at batches of one frame per wave: blocks of
4, 6 and 8 waves whose threads hold the next stage's image (D = N = 1 024:
17 pieces at 4 waves, the last a partial one, 12 at more), codebook chunks that are no multiple of the unrolled
step, a codebook read from memory, both summation orders, with and without
the reconstruction; channel-major input with ragged tiles; bit for bit."""

import re

import numpy as np
import pytest

from test_dac_gpu import _sha

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wpb", [4, 6, 8])
@pytest.mark.parametrize("T,D,N,channel_major,recon", [
    (1, 1024, 1024, False, False),
    (647, 1024, 1024, True, False),    # 162 blocks of 4 waves; the gather's last tile of 7 frames
    (65, 1024, 960, True, True),       # 15 chunks of codes
    (64, 1024, 1024, False, True),     # tinyBLAS order with recon: the copied image
    (132, 1024, 1024, True, False),    # tinyBLAS order, held image
    (5, 1024, 4096, False, False),     # codebook in memory
    (63, 256, 64, True, True),
])
def test_dac_one_frame_per_wave(monkeypatch, T, D, N, channel_major, recon, wpb):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle

    print(f"[gpu] dac one frame per wave T={T} D={D} N={N} cm={channel_major} recon={recon} waves={wpb}", flush=True)
    monkeypatch.setenv("AQ_DAC_FW", "1")
    monkeypatch.setenv("AQ_DAC_WPB", str(wpb))
    Q = 3
    cfg = dict(synth.dac_weights(91, Q, D, N, bias=True), x=synth.normal(91, 1, (T, D)), M=T, T=T, B=1, D=D, N=N, Q=Q)
    st = aqmi.DacStages(aqmi.Context(0), cfg["w_in"], cfg.get("b_in"), cfg["codebook"], cfg["w_out"], cfg.get("b_out"))
    x = torch.from_numpy(cfg["x"]).cuda()
    x = x.t().contiguous() if channel_major else x
    idx = torch.full((T, Q), -1, dtype=torch.int32, device="cuda")
    res = torch.empty((T, D), dtype=torch.float32, device="cuda")
    rec = torch.empty((T, D), dtype=torch.float32, device="cuda") if recon else None
    st.encode_ex(x, T, T, (D * T, 1, T) if channel_major else (D * T, D, 1), idx.data_ptr(), Q, res, rec)
    torch.cuda.synchronize()
    ref = Oracle().dac_rvq(cfg)
    assert np.array_equal(idx.cpu().numpy(), ref["idx"])
    assert _sha(res.cpu().numpy()) == _sha(ref["residual"])
    if recon:
        assert _sha(rec.cpu().numpy()) == _sha(ref["recon"])


@pytest.mark.parametrize("recon", [False, True])
def test_dac_held_pieces_follow_the_block(monkeypatch, capfd, recon):
    """Blocks that need no more than 12 pieces hold 12, whatever the frames per
    wave; wider blocks of one frame per wave hold 17 (tinyBLAS order with
    recon: the image is copied)."""
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle

    T, D, N, Q = 1100, 1024, 1024, 2   # a multiple of 4: the tinyBLAS order
    cfg = dict(synth.dac_weights(91, Q, D, N, bias=True), x=synth.normal(91, 1, (T, D)), M=T, T=T, B=1, D=D, N=N, Q=Q)
    st = aqmi.DacStages(aqmi.Context(0), cfg["w_in"], cfg.get("b_in"), cfg["codebook"], cfg["w_out"], cfg.get("b_out"))
    x = torch.from_numpy(cfg["x"]).cuda()
    idx = torch.full((T, Q), -1, dtype=torch.int32, device="cuda")
    rec = torch.empty((T, D), dtype=torch.float32, device="cuda") if recon else None
    capfd.readouterr()
    monkeypatch.setenv("AQ_DEBUG", "1")
    st.encode(x, T, idx, None, rec)
    torch.cuda.synchronize()
    held = {(int(fw), int(wpb)): int(pf) for fw, wpb, pf in
            re.findall(r"shape fw=(\d) wpb=(\d) pf=(\d+)", capfd.readouterr().err)}
    assert held[1, 4] == (0 if recon else 17)
    assert held[1, 6] == held[1, 8] == held[2, 8] == 12
    ref = Oracle().dac_rvq(cfg)
    assert np.array_equal(idx.cpu().numpy(), ref["idx"])
    if recon:
        assert _sha(rec.cpu().numpy()) == _sha(ref["recon"])


@pytest.mark.parametrize("M", [9, 2049, 4097, 5121])   # 3, 3, 5 and 6 waves per block, the last one of one frame
def test_outetts_waves_per_block(M):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle
    from test_hostloop_gpu import run_outetts

    print(f"[gpu] outetts waves per block M={M}", flush=True)
    cfg = synth.outetts_config(M)
    got = run_outetts(torch, aqmi.Context(0), cfg)
    want = Oracle().outetts_rvq(cfg)
    assert np.array_equal(got["idx"], want["idx"])
    assert _sha(got["residual"]) == _sha(want["residual"])


@pytest.mark.parametrize("Q", [1, 2, 3, 5, 8, 9, 17])   # one, two, four and eight stages' rows at once, with remainders
def test_dac_decode_stage_counts(Q):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import aqmi
    from aqmi import synth
    from oracle import Oracle

    print(f"[gpu] dac decode Q={Q}", flush=True)
    T, D, N = 37, 128, 64
    cfg = dict(synth.dac_weights(93, Q, D, N, bias=True), x=synth.normal(93, 1, (T, D)), M=T, T=T, B=1, D=D, N=N, Q=Q)
    st = aqmi.DacStages(aqmi.Context(0), cfg["w_in"], cfg.get("b_in"), cfg["codebook"], cfg["w_out"], cfg.get("b_out"))
    codes = np.random.default_rng(3).integers(0, N, (T, Q)).astype(np.int32)
    recon = Oracle().dac_rvq(cfg, codes)["recon"]   # teacher forced: the sum over these codes
    idx = torch.from_numpy(codes).cuda()
    out = torch.empty((T, D), dtype=torch.float32, device="cuda")
    st.decode(idx, out)
    assert _sha(out.cpu().numpy()) == _sha(recon)
    first = torch.from_numpy(synth.normal(93, 2, (T, D))).cuda()   # one stage added to what is there
    one = aqmi.DacStages(aqmi.Context(0), *(cfg[k][:1] for k in ("w_in", "b_in", "codebook", "w_out", "b_out")))
    z0 = torch.empty_like(out)
    one.decode(idx[:, :1].contiguous(), z0)
    want = first + z0
    one.decode_ex(idx.data_ptr(), Q, T, first, True)
    assert _sha(first.cpu().numpy()) == _sha(want.cpu().numpy())
    idx[T - 1, Q - 1] = N
    with pytest.raises(aqmi.AqError) as e:
        st.decode(idx, out)
    assert e.value.status == 3
