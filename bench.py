"""Throughput of the codec-quantizer hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload NAME]

A step is one pass of the RVQ encode over one batch of synthetic input
(generated by aqmi.synth with fixed seeds).  Inputs are
resident in HBM before the timed region; R input/output sets are rotated so
the live set exceeds the 256 MB Infinity Cache and every step streams from HBM.
Rank 0 prints one JSON line.

Timing
  value        frames encoded per second of wall clock over exactly K steps,
               bracketed by torch.cuda.synchronize() on both sides, with no
               events on the stream.
  roofline     algorithmic work per launch of the dominant kernel divided by
               its average duration, measured in a second pass of K steps:
               the library launches the kernel with hipExtLaunchKernelGGL's
               start and stop events (aq_ctx_set_timing), which time the
               kernel's own execution on the stream it runs on (the library
               runs on torch's current stream).  The Euclidean workloads whose
               step is one launch (the one-launch cascades) count all stages'
               work in that launch.
  cpu_baseline the reference's own ggml CPU backend (oracle/_ref, compiled
               from the reference sources) timed on this host's cores on a
               bounded sample of the same workload; graph compute only.
"""

from __future__ import annotations

import argparse
import json
import os
import pathlib
import sys
import time

import numpy as np

ROOT = pathlib.Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))
sys.path.insert(0, str(ROOT / "audio.cpp_amd"))

METRIC = "RVQ-encoded frames/sec at 1 MI355X; % of HBM or MFMA roofline"
HBM_PEAK_GBS = 8000.0
FP32_PEAK_TFLOPS = 157.3
# one fp32 FMA per lane and cycle: the rate without packed fp32 math, which
# this build leaves off
FP32_UNPACKED_PEAK_TFLOPS = FP32_PEAK_TFLOPS / 2
BF16_PEAK_TFLOPS = 2500.0
MALL_ROTATE_BYTES = 512 << 20


def log(msg: str):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


# ----------------------------------------------------------------- workloads

class DacRvq:
    """DAC cosine RVQ, 12 stages, 8 clips x 750 frames,
    D = 1024, codebooks 1024 x 8; outputs codes [M, 12] and the
    reconstructed latent [M, D]."""

    name = "dac_rvq_cfg1"
    kernel = "dac_encode_ms_kernel"
    cfg_id = 1

    def __init__(self, torch, aqmi, synth):
        self.torch = torch
        cfg = synth.make_config(self.cfg_id)
        self.cfg = cfg
        self.M, self.D, self.Q, self.N, self.T = cfg["x"].shape[0], cfg["D"], cfg["Q"], cfg["N"], cfg["T"]
        self.ctx = aqmi.Context(0)
        self.st = aqmi.DacStages(self.ctx, cfg["w_in"], cfg["b_in"], cfg["codebook"], cfg["w_out"], cfg["b_out"])
        per_set = self.M * self.D * 4 * 2 + self.M * self.Q * 4
        self.R = max(1, -(-MALL_ROTATE_BYTES // per_set))
        x = torch.from_numpy(cfg["x"]).cuda()
        self.x = [x] + [x.clone() for _ in range(self.R - 1)]
        self.idx = [torch.empty((self.M, self.Q), dtype=torch.int32, device="cuda") for _ in range(self.R)]
        self.rec = [torch.empty((self.M, self.D), dtype=torch.float32, device="cuda") for _ in range(self.R)]
        self.live_bytes = per_set * self.R

    def step(self, k: int):
        r = k % self.R
        self.st.encode(self.x[r], self.T, self.idx[r], None, self.rec[r])

    # Algorithmic work of one launch (one kernel runs all 12 stages for all M
    # frames).  Per frame-stage: in-projection 2*D*8, cosine scores 2*8*N,
    # out-projection 2*8*D, residual update D  ->  50 176 FLOP at D = N = 1024.
    def flops_per_frame(self) -> float:
        return self.Q * (2 * self.D * 8 + 2 * 8 * self.N + 2 * 8 * self.D + self.D)

    def hbm_bytes_per_frame(self) -> float:
        # read x, write recon, write Q codes (the cascade stays on chip).
        return self.D * 4 * 2 + self.Q * 4

    def flops_per_launch(self) -> float:
        return self.flops_per_frame() * self.M

    # Algorithmic HBM bytes of a per-stage design (the accounting the
    # workload's roofline is quoted in): per frame-stage, read and write the
    # D-float residual and write one code -> 8 196 B, x 12 stages = 98 352 B.
    def algorithmic_bytes_per_frame(self) -> float:
        return self.Q * (2 * self.D * 4 + 4)

    # The part of the work that runs on the VALU in exact-order fp32: the
    # in-projection's FMA chains and the residual / reconstruction updates;
    # the approximate scores run on fp16 matrix cores (split operands).
    def valu_flops_per_frame(self) -> float:
        return self.Q * (2 * self.D * 8 + 2 * self.D)

    def roofline(self, avg_launch_s: float) -> dict:
        achieved = self.algorithmic_bytes_per_frame() * self.M / avg_launch_s / 1e9
        fp32 = self.flops_per_frame() * self.M / avg_launch_s / 1e12
        valu = self.valu_flops_per_frame() * self.M / avg_launch_s / 1e12
        return {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": measured_traffic(self.kernel, self.name),
                "note": f"achieved = {self.algorithmic_bytes_per_frame():.0f} algorithmic B/frame (per-stage residual "
                        f"read + write + code, {self.Q} stages) x {self.M} frames / kernel time; the fused kernel "
                        f"keeps the cascade on chip and moves {self.hbm_bytes_per_frame():.0f} B/frame "
                        f"({self.hbm_bytes_per_frame() * self.M / avg_launch_s / 1e9:.1f} GB/s); "
                        f"algorithmic work {fp32:.2f} TFLOP/s, of which the cosine scores run on fp16 matrix cores",
                # the exact-order fp32 part on the VALU (packed math off)
                "binding": {"resource": "valu", "achieved": round(valu, 2), "peak": FP32_UNPACKED_PEAK_TFLOPS,
                            "unit": "TFLOP/s", "frac": round(valu / FP32_UNPACKED_PEAK_TFLOPS, 4),
                            "note": "in-projection FMA chains and residual / reconstruction updates only"}}

    def parity(self) -> dict:
        g = np.load(ROOT / "tests" / "golden" / "dac_cfg1.npz")
        got = self.idx[0].cpu().numpy()
        want = g["idx"].astype(np.int32)
        return {"idx_agree": float((got == want).mean()), "fixture": "tests/golden/dac_cfg1.npz",
                **near_ties("dac_cfg1.npz")}

    def config(self) -> dict:
        return {"workload": "BASELINE configs[1]: DAC cosine RVQ", "frames": self.M, "clips": self.M // self.T,
                "clip_len": self.T, "latent_dim": self.D, "stages": self.Q, "codebook": [self.N, 8],
                "outputs": "codes int32 [M,12] + reconstructed latent fp32 [M,1024]",
                "rotating_sets": self.R, "live_MB": round(self.live_bytes / 2**20, 1)}

    def cpu_baseline(self, threads: int, budget_s: float = 12.0) -> dict:
        from oracle import Ref

        ref = Ref()
        ref.dac_rvq(self.cfg, threads=threads, recon=True)        # warm-up
        times = []
        t0 = time.perf_counter()
        while len(times) < 7 and (time.perf_counter() - t0) < budget_s:
            times.append(ref.dac_rvq(self.cfg, threads=threads, recon=True)["ms"])
        ms = float(np.median(times))
        return {"value": round(self.M / (ms / 1e3), 1), "unit": "frames/s", "cores": threads, "kind": "reference",
                "sample": f"full config 1 ({self.M} frames x {self.Q} stages), ggml CPU graph compute only, "
                          f"median of {len(times)} runs, ggml build {ref.isa}, {_cpu_model()}"}


class EuclidRvq:
    """Euclidean VQ / RVQ on fp16 matrix cores with exact fp32 re-ranking.
    Subclasses fix the BASELINE config, the reference recipe and the
    outputs."""

    kernel = "euclid_sweep_kernel"
    cfg_id = 2
    recipe_name = "OMNIVOICE"
    cb_key = "codebook"
    cb_type = 0
    topk = 0
    want_dist = False
    fixture = "mimi_cfg2.npz"
    cpu_rows = 4800

    def __init__(self, torch, aqmi, synth):
        self.torch = torch
        cfg = synth.make_config(self.cfg_id)
        self.cfg = cfg
        self.M, self.K, self.Q, self.N = cfg["M"], cfg["K"], cfg["Q"], cfg["N"]
        self.ctx = aqmi.Context(0)
        self.cbs = aqmi.Codebooks(self.ctx, cfg[self.cb_key], getattr(aqmi, self.recipe_name), self.cb_type)
        T = max(self.topk, 1)
        per_set = self.M * self.K * 4 + self.M * self.Q * 4 * (1 + (1 if self.want_dist else 0) + 2 * self.topk)
        self.R = max(1, -(-MALL_ROTATE_BYTES // per_set))
        x = torch.from_numpy(cfg["x"]).cuda()
        self.x = [x] + [x.clone() for _ in range(self.R - 1)]
        dev = dict(device="cuda")
        self.idx = [torch.empty((self.M, self.Q), dtype=torch.int32, **dev) for _ in range(self.R)]
        self.dist = [torch.empty((self.M, self.Q), dtype=torch.float32, **dev) if self.want_dist else None
                     for _ in range(self.R)]
        self.tki = [torch.empty((self.M, self.Q, T), dtype=torch.int32, **dev) if self.topk else None
                    for _ in range(self.R)]
        self.tkd = [torch.empty((self.M, self.Q, T), dtype=torch.float32, **dev) if self.topk else None
                    for _ in range(self.R)]
        self.live_bytes = per_set * self.R

    def step(self, k: int):
        r = k % self.R
        self.cbs.encode(self.x[r], self.idx[r], None, self.dist[r], self.topk, self.tki[r], self.tkd[r])

    # stages per timed launch: 1 for the per-stage pipeline (the timed launch
    # is the sweep), Q for the one-launch cascades (set by one_launch())
    stages_per_launch = 1

    def one_launch(self):
        """The step ran as one timed launch for all stages: the one-launch
        cascade (residual in LDS at K = 256)."""
        self.stages_per_launch = self.Q
        self.kernel = "euclid_narrow_kernel" if self.K == 256 else "euclid_cascade_kernel"

    def flops_per_launch(self) -> float:
        # the distance contraction of one stage is 2 * N * K per frame
        return 2.0 * self.N * self.K * self.M * self.stages_per_launch

    def roofline(self, avg_launch_s: float, step_s: float | None = None) -> dict:
        achieved = self.flops_per_launch() / avg_launch_s / 1e12
        if self.stages_per_launch > 1:
            note = (f"dominant kernel = the one-launch cascade (fp16 MFMA sweep, select and residual update of all "
                    f"{self.Q} stages): {self.Q} x {self.M} x {self.N} x {self.K} MACs (2 FLOP each) per launch; "
                    "peak = dense fp16 MFMA")
        else:
            note = (f"dominant kernel = the fp16 MFMA sweep, one launch per stage: {self.M} x {self.N} x {self.K} MACs "
                    "(2 FLOP each); peak = dense fp16 MFMA")
        if step_s:
            whole = 2.0 * self.N * self.K * self.M * self.Q / step_s / 1e12
            note += (f"; whole step incl. every kernel: {whole:.1f} TFLOP/s "
                     f"({whole / BF16_PEAK_TFLOPS:.3f} of peak)")
        if self.cb_type:
            # the codebook is stored as int8 blocks: the same work against
            # the dense int8 matrix peak
            note += f"; against the dense int8 peak ({INT8_PEAK_TOPS:.0f} TOP/s): {achieved / INT8_PEAK_TOPS:.3f}"
        return {"bound": "mfma", "achieved": round(achieved, 2), "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                "frac": round(achieved / BF16_PEAK_TFLOPS, 4), "traffic": measured_traffic(self.kernel, self.name),
                "note": note}

    def parity(self) -> dict:
        path = ROOT / "tests" / "golden" / self.fixture
        g = np.load(path)
        got = self.idx[0].cpu().numpy()
        want = g["idx"].astype(np.int32).reshape(got.shape)
        return {"idx_agree": float((got == want).mean()), "fixture": str(path.relative_to(ROOT)),
                **near_ties(self.fixture),
                **({"verified_frames_per_stage": self.cbs.failures().tolist(),
                    "recomputed_frames_per_stage": self.cbs.exact_scans().tolist()}
                   if self.stages_per_launch > 1 else
                   {"refined_frames_per_stage": self.cbs.failures().tolist(),
                    "exact_scan_frames_per_stage": self.cbs.exact_scans().tolist()})}

    def outputs(self) -> str:
        out = f"codes int32 [{self.M},{self.Q}]"
        if self.want_dist:
            out += f" + distance fp32 [{self.M},{self.Q}]"
        if self.topk:
            out += f" + top-{self.topk} codes and distances per stage"
        return out

    def config(self) -> dict:
        return {"workload": self.workload, "frames": self.M, "dim": self.K, "stages": self.Q,
                "codebook": [self.N, self.K], "codebook_type": "q8_0" if self.cb_type else "f32",
                "recipe": self.recipe_name.lower(), "outputs": self.outputs(),
                "rotating_sets": self.R, "live_MB": round(self.live_bytes / 2**20, 1)}

    def _ref_call(self, ref, sample, threads):
        return ref.euclid_rvq(sample, threads=threads)

    def cpu_baseline(self, threads: int, budget_s: float = 12.0) -> dict:
        from oracle import Ref

        ref = Ref()
        rows = self.cpu_rows
        sample = dict(self.cfg, x=self.cfg["x"][:rows], M=rows)
        self._ref_call(ref, dict(sample, x=sample["x"][:rows // 10], M=rows // 10), threads)   # warm-up
        times = []
        t0 = time.perf_counter()
        while len(times) < 5 and (time.perf_counter() - t0) < budget_s:
            times.append(self._ref_call(ref, sample, threads)["ms"])
        ms = float(np.median(times))
        return {"value": round(rows / (ms / 1e3), 1), "unit": "frames/s", "cores": threads, "kind": "reference",
                "sample": f"first {rows} of {self.M} frames x {self.Q} stage(s), ggml CPU graph compute only "
                          f"({self.recipe_name.lower()} recipe), median of {len(times)} runs, ggml build {ref.isa}, "
                          f"{_cpu_model()}"}


class MimiRvq(EuclidRvq):
    """Mimi-style Euclidean RVQ, 8 codebooks 2048 x 256,
    48 000 frames of dim 256; argmin |x - c|^2 as |c|^2 - 2 x.c (the OmniVoice
    recipe); int32 codes [48000, 8]."""

    name = "mimi_rvq_cfg2"
    workload = "BASELINE configs[2]: Mimi-style Euclidean RVQ"


class KMeans(EuclidRvq):
    """semantic k-means, 200 000 frames x 768 against
    16 384 centroids, one stage; code plus min distance (the Higgs recipe,
    whose -logit is |r|^2 + |c|^2 - 2 c.r)."""

    name = "kmeans_cfg3"
    workload = "BASELINE configs[3]: k-means tokenisation"
    cfg_id = 3
    recipe_name = "HIGGS"
    want_dist = True
    fixture = "kmeans_cfg3.npz"
    cpu_rows = 2000

    def _ref_call(self, ref, sample, threads):
        return ref.higgs_rvq(sample, threads=threads)


class Q8Rvq(EuclidRvq):
    """the Mimi RVQ with GGUF Q8_0 codebooks (Higgs
    recipe: the query is quantised to Q8_0 with x86 rounding, integer block
    dots), top-4 codes and distances per stage."""

    name = "q8_rvq_cfg4"
    workload = "BASELINE configs[4]: Q8_0-codebook Mimi RVQ with top-4"
    cfg_id = 4
    recipe_name = "HIGGS"
    cb_key = "codebook_q8"
    cb_type = 1
    topk = 4
    want_dist = True
    fixture = "q8_cfg4.npz"

    def _ref_call(self, ref, sample, threads):
        return ref.higgs_rvq(sample, topk=4, threads=threads)


FP64_PEAK_TFLOPS = 78.6
INT8_PEAK_TOPS = 5000.0


class OuteTtsRvq:
    """OuteTTS DAC host-loop quantizer (not a BASELINE config; the shapes of
    community_models/outetts/dac.cpp:376-456): 6 000 frames of the D = 1024
    latent, 2 stages of 1024 x 8 codes, fp32 sequential arithmetic; outputs
    the codes, as the reference does."""

    name = "outetts_rvq"
    kernel = "outetts_encode_kernel"
    fixture = "outetts_bench.npz"

    def __init__(self, torch, aqmi, synth):
        self.torch = torch
        cfg = synth.outetts_config(6000)
        self.cfg = cfg
        self.M, self.D, self.Q, self.N = cfg["M"], cfg["D"], cfg["Q"], cfg["N"]
        self.ctx = aqmi.Context(0)
        self.st = aqmi.DacStages(self.ctx, cfg["w_in"], cfg["b_in"], cfg["codebook"], cfg["w_out"], cfg["b_out"],
                                 recipe=aqmi.DAC_OUTETTS)
        per_set = self.M * self.D * 4 + self.M * self.Q * 4
        self.R = max(1, -(-MALL_ROTATE_BYTES // per_set))
        x = torch.from_numpy(cfg["x"]).cuda()
        self.x = [x] + [x.clone() for _ in range(self.R - 1)]
        self.idx = [torch.empty((self.M, self.Q), dtype=torch.int32, device="cuda") for _ in range(self.R)]
        self.live_bytes = per_set * self.R

    def step(self, k: int):
        r = k % self.R
        self.st.encode(self.x[r], self.M, self.idx[r])

    # per frame-stage: in-projection 2*8*D, distances 3*8*N, out-projection
    # 2*8*D, residual update D
    def flops_per_frame(self) -> float:
        return self.Q * (2 * 8 * self.D + 3 * 8 * self.N + 2 * 8 * self.D + self.D)

    def roofline(self, avg_launch_s: float) -> dict:
        per_frame = self.Q * (2 * self.D * 4 + 4)
        achieved = per_frame * self.M / avg_launch_s / 1e9
        fp32 = self.flops_per_frame() * self.M / avg_launch_s / 1e12
        return {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": measured_traffic(self.kernel, self.name),
                "note": f"per-stage accounting as the DAC workload: {per_frame} B/frame x {self.M} frames / kernel "
                        f"time; the kernel keeps the residual in LDS; fp32 work {fp32:.2f} TFLOP/s of "
                        f"{FP32_PEAK_TFLOPS} (sequential chains, products rounded before the add)"}

    def parity(self) -> dict:
        path = ROOT / "tests" / "golden" / self.fixture
        got = self.idx[0].cpu().numpy()
        want = np.load(path)["idx"].astype(np.int32)
        return {"idx_agree": float((got == want).mean()), "fixture": str(path.relative_to(ROOT))}

    def config(self) -> dict:
        return {"workload": "OuteTTS DAC host-loop RVQ (dac.cpp:376-456 shapes; not a BASELINE config)",
                "frames": self.M, "latent_dim": self.D, "stages": self.Q, "codebook": [self.N, 8],
                "outputs": f"codes int32 [{self.M},{self.Q}]", "rotating_sets": self.R,
                "live_MB": round(self.live_bytes / 2**20, 1)}

    def cpu_baseline(self, threads: int, budget_s: float = 12.0) -> dict:
        from oracle import Ref

        ref = Ref()
        ref.outetts_rvq(self.cfg, threads=threads)   # warm-up
        times = []
        t0 = time.perf_counter()
        while len(times) < 5 and (time.perf_counter() - t0) < budget_s:
            times.append(ref.outetts_rvq(self.cfg, threads=threads, timed=True)[1])
        ms = float(np.median(times))
        return {"value": round(self.M / (ms / 1e3), 1), "unit": "frames/s", "cores": threads, "kind": "reference",
                "sample": f"full workload ({self.M} frames x {self.Q} stages), the reference's quantize_reference "
                          f"(OpenMP), median of {len(times)} runs, {_cpu_model()}"}


class MossRvq:
    """MOSS RLFQ quantizer (not a BASELINE config; MOSS-Audio-Tokenizer-v2
    shapes, audio_tokenizer_quantizer.cpp): 6 000 frames of the 768-channel
    encoder latent, fp64 input projection to 512 and 12 stages of 1024 x 8
    codes; outputs the codes, as the reference does."""

    name = "moss_rvq"
    kernels = ("moss_input_kernel", "moss_cascade_kernel")
    fixture = "moss_bench.npz"

    def __init__(self, torch, aqmi, synth):
        self.torch = torch
        cfg = synth.moss_config(6000)
        self.cfg = cfg
        self.M, self.C, self.R_, self.Q, self.N = cfg["M"], cfg["C"], cfg["R"], cfg["Q"], cfg["N"]
        self.ctx = aqmi.Context(0)
        f = synth.moss_fold(cfg)
        self.q = aqmi.MossQuantizer(self.ctx, f["w_ip"], cfg["ip_b"], f["w_in"], cfg["in_b"], cfg["codebook"],
                                    f["w_out"], cfg["out_b"])
        per_set = self.M * self.C * 4 + self.M * self.Q * 4
        self.R = max(1, -(-MALL_ROTATE_BYTES // per_set))
        h = torch.from_numpy(cfg["hidden"]).cuda()
        self.h = [h] + [h.clone() for _ in range(self.R - 1)]
        self.idx = [torch.empty((self.M, self.Q), dtype=torch.int32, device="cuda") for _ in range(self.R)]
        self.live_bytes = per_set * self.R
        self.kernel = self.kernels[1]

    def step(self, k: int):
        r = k % self.R
        self.q.encode(self.h[r], self.idx[r])

    def split(self, kernel_ms):
        """Per-kernel mean launch times (the library times both launches)."""
        per = np.asarray(kernel_ms).reshape(-1, len(self.kernels))
        return {k: float(per[:, i].mean()) / 1e3 for i, k in enumerate(self.kernels)}

    def flops_per_frame(self, kernel: str) -> float:
        if kernel == "moss_input_kernel":
            return 2.0 * self.C * self.R_
        # per stage: in-projection 2*8*R, dots 2*8*N, out-projection 2*8*R, residual R
        return self.Q * (2 * 8 * self.R_ + 2 * 8 * self.N + 2 * 8 * self.R_ + self.R_)

    def roofline(self, avg_launch_s: float, per_kernel: dict | None = None) -> dict:
        achieved = self.flops_per_frame(self.kernel) * self.M / avg_launch_s / 1e12
        note = (f"fp64 work of {self.kernel} per launch / its time; peak = MI355X fp64 ({FP64_PEAK_TFLOPS} TFLOP/s, "
                "vector and matrix); exact-order sums are VALU chains, not MFMA")
        if per_kernel:
            note += "; per launch: " + ", ".join(f"{k} {v * 1e6:.1f} us" for k, v in per_kernel.items())
        return {"bound": "mfma", "achieved": round(achieved, 3), "peak": FP64_PEAK_TFLOPS, "unit": "TFLOP/s",
                "frac": round(achieved / FP64_PEAK_TFLOPS, 4), "traffic": measured_traffic(self.kernel, self.name),
                "note": note}

    def parity(self) -> dict:
        path = ROOT / "tests" / "golden" / self.fixture
        got = self.idx[0].cpu().numpy()
        want = np.load(path)["idx"].astype(np.int32)
        return {"idx_agree": float((got == want).mean()), "fixture": str(path.relative_to(ROOT))}

    def config(self) -> dict:
        return {"workload": "MOSS RLFQ quantizer (MOSS-Audio-Tokenizer-v2 shapes; not a BASELINE config)",
                "frames": self.M, "code_dim": self.C, "rvq_dim": self.R_, "stages": self.Q,
                "codebook": [self.N, 8], "outputs": f"codes int32 [{self.M},{self.Q}]", "rotating_sets": self.R,
                "live_MB": round(self.live_bytes / 2**20, 1)}

    def cpu_baseline(self, threads: int, budget_s: float = 12.0) -> dict:
        from oracle import Ref

        ref = Ref()
        times = []
        t0 = time.perf_counter()
        while len(times) < 5 and (time.perf_counter() - t0) < budget_s:
            times.append(ref.moss_encode_timed(self.cfg, threads=threads)[1])
        ms = float(np.median(times))
        return {"value": round(self.M / (ms / 1e3), 1), "unit": "frames/s", "cores": threads, "kind": "reference",
                "sample": f"full workload ({self.M} frames x {self.Q} stages), the reference's "
                          f"MossAudioTokenizerQuantizer::encode (OpenMP; constructor outside the clock), median of "
                          f"{len(times)} runs, {_cpu_model()}"}


WORKLOADS = {"dac_rvq": DacRvq, "mimi_rvq": MimiRvq, "kmeans": KMeans, "q8_rvq": Q8Rvq,
             "outetts_rvq": OuteTtsRvq, "moss_rvq": MossRvq}


def near_ties(fixture: str) -> dict:
    """Near-tie accounting of a golden fixture (tests/golden/near_ties.json,
    written by tests/golden/near_ties.py): frame-stages whose fp64
    best/second distance gap is <= 1e-5 relative on the reference's path."""
    path = ROOT / "tests" / "golden" / "near_ties.json"
    if not path.exists():
        return {}
    entry = json.loads(path.read_text()).get(fixture)
    if not entry:
        return {}
    return {"near_ties": int(sum(entry["near_ties_per_stage"])), "frame_stages": entry["frame_stages"],
            "near_tie_rule": "fp64 gap_rel <= 1e-5 on the reference's residual path",
            "fp64_argmin_differs_outside_near_ties": int(sum(entry["argmin_differs_outside_ties"]))}


def host_cpu() -> dict:
    """The host's CPU as this process sees it."""
    info = {"model": _cpu_model(), "nproc": len(os.sched_getaffinity(0)), "cpu_count": os.cpu_count()}
    try:
        quota, period = open("/sys/fs/cgroup/cpu.max").read().split()
        if quota != "max":
            info["cgroup_cpus"] = round(int(quota) / int(period), 2)
    except (OSError, ValueError):
        pass
    return info


def measured_traffic(kernel: str, workload: str):
    """HBM bytes per launch of `kernel` on `workload` from the committed
    rocprofv3 --pmc summary (FETCH_SIZE and WRITE_SIZE, each scaled by a
    calibration copy); None when that pair has not been measured."""
    path = ROOT / "profiles" / "traffic.json"
    if not path.exists():
        return None
    entry = json.loads(path.read_text()).get(f"{kernel}@{workload}")
    return None if entry is None else entry["bytes_per_launch"]


def _cpu_model() -> str:
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown CPU"


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--workload", default="dac_rvq", choices=sorted(WORKLOADS))
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-threads", type=int, default=0, help="CPU baseline threads (default: nproc)")
    ap.add_argument("--no-secondary", action="store_true", help="skip the configs[2] block of the default run")
    ap.add_argument("--calibrate-copy-mb", type=int, default=0,
                    help="first run a plain device copy of this many MiB 5 times (HBM counter calibration)")
    args = ap.parse_args()

    if args.gpus != 1:
        print(f"bench.py measures one GPU only: this build has no multi-GPU path (asked for --gpus {args.gpus}).",
              file=sys.stderr)
        sys.exit(2)

    import torch

    import aqmi
    from aqmi import synth

    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(1)

    if args.calibrate_copy_mb:
        n = args.calibrate_copy_mb * (1 << 20) // 4
        src = torch.ones(n, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(5):
            dst.copy_(src)
        torch.cuda.synchronize()
        log(f"calibration copy: 5 x {args.calibrate_copy_mb} MiB read + write")
        del src, dst

    threads = args.cpu_threads or len(os.sched_getaffinity(0))
    out = measure(WORKLOADS[args.workload], torch, aqmi, synth, args.steps, args.warmup,
                  None if args.no_cpu_baseline else threads)
    out = {"metric": METRIC, **out}
    if args.workload == "dac_rvq" and not args.no_secondary:
        # BASELINE configs[2] (the north star's Mimi target), timed in the same run
        sec = measure(MimiRvq, torch, aqmi, synth, min(args.steps, 100), min(args.warmup, 10),
                      None if args.no_cpu_baseline else threads)
        out["secondary"] = {k: sec[k] for k in ("value", "unit", "steps", "ms_per_step", "config", "kernel",
                                                "kernel_avg_us", "kernel_launches_per_step", "roofline", "parity",
                                                "cpu_baseline") if k in sec}
    print(json.dumps(out), flush=True)


def measure(cls, torch, aqmi, synth, K: int, W: int, threads: int | None) -> dict:
    """Warm-up, throughput over exactly K steps, kernel durations over K more
    steps, parity and (threads given) the CPU baseline of one workload."""
    log(f"workload {cls.__name__}: generating inputs")
    wl = cls(torch, aqmi, synth)
    log(f"warmup {W}")
    for k in range(W):
        wl.step(k)
    torch.cuda.synchronize()

    # Throughput: exactly K steps with nothing else on the stream.
    log(f"timing {K} steps")
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(K):
        wl.step(W + k)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    # Kernel durations: the same K steps again with HIP events around every
    # launch (the events add gaps between launches, so this pass gives the
    # roofline and the step log line, not the throughput).
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(K)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(K)]
    log(f"timing {K} steps with per-launch events")
    wl.ctx.set_timing(True)
    torch.cuda.synchronize()
    for k in range(K):
        starts[k].record()
        wl.step(W + K + k)
        ends[k].record()
    torch.cuda.synchronize()
    kernel_ms = wl.ctx.read_timing()
    wl.ctx.set_timing(False)
    step_ms = [s.elapsed_time(e) for s, e in zip(starts, ends)]
    per_kernel = None
    if hasattr(wl, "split"):
        # workloads with several timed launches per step: the dominant one
        per_kernel = wl.split(kernel_ms)
        wl.kernel = max(per_kernel, key=per_kernel.get)
        avg_launch_s = per_kernel[wl.kernel]
        kernel_ms = np.asarray(kernel_ms).reshape(-1, len(per_kernel))[:, list(per_kernel).index(wl.kernel)]
    else:
        avg_launch_s = float(np.mean(kernel_ms)) / 1e3
    if isinstance(wl, EuclidRvq) and len(kernel_ms) == K and wl.Q > 1:
        wl.one_launch()
    log(f"wall {wall * 1e3:.3f} ms, step mean {np.mean(step_ms) * 1e3:.2f} us; {len(kernel_ms)} launches of "
        f"{wl.kernel}: mean {avg_launch_s * 1e6:.2f} us, min {kernel_ms.min() * 1e3:.2f} us, "
        f"max {kernel_ms.max() * 1e3:.2f} us")

    # One extra (untimed) step on set 0 for the parity summary.
    wl.step(0)
    torch.cuda.synchronize()
    parity = wl.parity()

    out = {
        "value": round(wl.M * K / wall, 1), "unit": "frames/s", "n_gpus": 1, "steps": K,
        "warmup": W, "ms_per_step": round(wall * 1e3 / K, 5), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic (aqmi.synth, seeded)",
        "config": wl.config(), "kernel": wl.kernel, "kernel_avg_us": round(avg_launch_s * 1e6, 3),
        "kernel_launches_per_step": round(len(kernel_ms) / K, 2),
        "roofline": (wl.roofline(avg_launch_s, wall / K) if isinstance(wl, EuclidRvq)
                     else wl.roofline(avg_launch_s, per_kernel) if per_kernel else wl.roofline(avg_launch_s)),
        "parity": parity,
    }
    if threads:
        log(f"cpu baseline on {threads} threads")
        try:
            out["cpu_baseline"] = dict(wl.cpu_baseline(threads), host=host_cpu())
        except (FileNotFoundError, OSError) as e:
            out["cpu_baseline"] = {"value": None, "unit": "frames/s", "cores": threads, "kind": "reference",
                                   "sample": f"unavailable: {e}", "host": host_cpu()}
    del wl
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return out


if __name__ == "__main__":
    main()
