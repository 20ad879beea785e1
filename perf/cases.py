"""The quantizer calls that a codec or tokeniser makes, as cases to measure.

Each case names a kind of call (KINDS), its sizes and its options; prepare()
builds the weights and inputs of a seed on the GPU, run() makes the call
through the aqmi binding, and exact() restates it in 64 bits with torch.
Shapes are those of the models the library serves; inputs and codebooks are
normal as in aqmi.synth.  Every result is specified bit for bit (the
reference's fp32 operation order), so the tolerance is "exact".
"""

import functools
import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "audio.cpp_amd"))

import aqmi  # noqa: E402
from aqmi import synth  # noqa: E402

DEV = "cuda"
RECIPES = {"omnivoice": aqmi.OMNIVOICE, "higgs": aqmi.HIGGS, "direct": aqmi.DIRECT}


def listed():
    return [
        # The smallest call: a 10 s voice prompt through the Qwen3-TTS speech
        # tokeniser (12.5 frames/s), 1 semantic + 15 acoustic EMA codebooks
        # of 2048 x 256 on the encoder's channel-major latents.
        dict(name="qwen3_clip", kind="qwen3", T=125, stages=16, N=2048, K=256),
        # A corpus batch through a Mimi-style codec: codes only.
        dict(name="mimi_batch", kind="rvq", B=1, T=48000, Q=8, N=2048, K=256, recipe="omnivoice", q8=False, topk=0,
             dist=False, residual=False, channel_major=False),
        # The same batch against Q8_0 codebooks with the four best codes and
        # their distances per stage (beam or soft-label use).
        dict(name="mimi_q8_top4", kind="rvq", B=1, T=48000, Q=8, N=2048, K=256, recipe="higgs", q8=True, topk=4,
             dist=True, residual=False, channel_major=False),
        # Semantic k-means tokens of one 30 s clip (50 frames/s, ragged end).
        dict(name="kmeans_clip", kind="rvq", B=1, T=1499, Q=1, N=16384, K=768, recipe="higgs", q8=False, topk=0,
             dist=True, residual=False, channel_major=False),
        # The largest call: k-means tokenisation of about 67 minutes.
        dict(name="kmeans_corpus", kind="rvq", B=1, T=200000, Q=1, N=16384, K=768, recipe="higgs", q8=False, topk=0,
             dist=True, residual=False, channel_major=False),
        # A 10 s voice prompt (25 frames/s) through the OmniVoice acoustic
        # quantizer: per-stage projections, fp32 weights, channel-major.
        dict(name="omnivoice_clip", kind="projected", B=1, T=250, H=1024, K=64, N=1024, Q=8, recipe="omnivoice",
             cb_q8=False, proj_q8=False, residual=False, channel_major=True),
        # A batch of 30 s clips through the Higgs quantizer stored as Q8_0.
        dict(name="higgs_q8_batch", kind="projected", B=8, T=750, H=1024, K=64, N=1024, Q=8, recipe="higgs",
             cb_q8=True, proj_q8=True, residual=True, channel_major=True),
        # A 30 s voice prompt (21.5 frames/s) through Fish Audio's quantizer:
        # one 4096-code stage chained with eight 1024-code stages.
        dict(name="fish_clip", kind="fish", B=1, T=647, D=1024, N0=4096, N=1024, Q=8, recon=False),
        # A batch of 10 s clips through the 12-stage DAC: codes and latent.
        dict(name="dac_batch", kind="dac", B=8, T=750, D=1024, N=1024, Q=12, recon=True, residual=False,
             channel_major=False),
        # A speaker reference through the OuteTTS DAC quantizer (14 s).
        dict(name="outetts_clip", kind="outetts", T=1046, D=1024, N=1024, Q=2),
        # A batch through the MOSS audio tokeniser's fp64 quantizer.
        dict(name="moss_batch", kind="moss", T=6000, C=768, R=512, N=1024, Q=12),
        # The way back: 60 s of generated Fish codes to the latent.
        dict(name="fish_decode", kind="decode", family="fish", T=1292, D=1024, N0=4096, N=1024, Q=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _flag(rng):
    return rng.random() < 0.5


def draw(rng):
    kind = rng.choice(("qwen3", "rvq", "q8", "kmeans", "projected", "fish", "dac", "outetts", "moss", "decode"))
    if kind == "qwen3":
        return dict(kind="qwen3", T=_log_int(rng, 20, 4000), stages=rng.choice((8, 16)), N=2048, K=256)
    if kind in ("rvq", "q8"):
        q8, B = kind == "q8", rng.choice((1, 1, 2, 5, 8))
        T = max(1, _log_int(rng, 100, 48000) // B)
        recipe = "higgs" if q8 else rng.choice(("omnivoice", "higgs", "direct"))
        return dict(kind="rvq", B=B, T=T, Q=rng.choice((4, 8)), N=rng.choice((1024, 2048)), K=256, recipe=recipe,
                    q8=q8, topk=rng.choice((0, 1, 4)) if q8 else 0, dist=q8 or _flag(rng), residual=_flag(rng),
                    channel_major=_flag(rng))
    if kind == "kmeans":
        return dict(kind="rvq", B=1, T=_log_int(rng, 100, 180000), Q=1, N=rng.choice((1024, 2048, 4096, 16384)),
                    K=rng.choice((512, 768)), recipe=rng.choice(("higgs", "omnivoice", "direct")), q8=False, topk=0,
                    dist=_flag(rng), residual=False, channel_major=False)
    if kind == "projected":
        recipe, B = rng.choice(("omnivoice", "higgs")), rng.choice((1, 1, 2, 8))
        T = max(2, _log_int(rng, 50, 6000) // B)
        q8 = recipe == "higgs" and _flag(rng)
        return dict(kind="projected", B=B, T=T, H=1024, K=64, N=1024, Q=8, recipe=recipe, cb_q8=q8, proj_q8=q8,
                    residual=_flag(rng), channel_major=_flag(rng))
    if kind == "fish":
        return dict(kind="fish", B=rng.choice((1, 2)), T=_log_int(rng, 40, 2600), D=1024, N0=4096, N=1024, Q=8,
                    recon=_flag(rng))
    if kind == "dac":
        B = rng.choice((1, 1, 2, 5, 8))
        T = max(1, _log_int(rng, 40, 6000) // B)
        return dict(kind="dac", B=B, T=T, D=rng.choice((512, 1024)), N=1024, Q=rng.choice((1, 4, 9, 12)),
                    recon=_flag(rng), residual=_flag(rng), channel_major=_flag(rng))
    if kind == "outetts":
        return dict(kind="outetts", T=_log_int(rng, 75, 6000), D=1024, N=1024, Q=2)
    if kind == "moss":
        return dict(kind="moss", T=_log_int(rng, 60, 6000), C=768, R=512, N=1024, Q=rng.choice((8, 12)))
    family, T = rng.choice(("fish", "rvq", "moss")), _log_int(rng, 40, 6000)
    if family == "fish":
        return dict(kind="decode", family="fish", T=T, D=1024, N0=4096, N=1024, Q=8)
    if family == "rvq":
        return dict(kind="decode", family="rvq", T=T, K=256, N=2048, Q=rng.choice((8, 16)))
    return dict(kind="decode", family="moss", T=T, C=768, R=512, N=1024, Q=12)


def tolerance(case):
    return "exact"


# ---- inputs ------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _context():
    """A program keeps one context per thread."""
    return aqmi.Context(0)


class _Values:
    """Normal, uniform and whole values of one seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV) * std

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(shape, generator=self.g, device=DEV)

    def codes(self, n, *shape):
        return torch.randint(0, n, shape, generator=self.g, device=DEV, dtype=torch.int32)

    def frames(self, case, width):
        """[B, C, T] as an encoder graph leaves it, or [B*T, C]."""
        B, T = case.get("B", 1), case["T"]
        return self.normal(B, width, T) if case.get("channel_major") else self.normal(B * T, width)

    def q8_blocks(self, *shape):
        """Random block_q8_0 rows as raw bytes [..., K/32, 34]."""
        lead = shape[:-1] + (shape[-1] // 32,)
        d = self.uniform(1e-3, 1e-2, *lead, 1).half()
        q = torch.randint(-127, 128, lead + (32,), generator=self.g, device=DEV, dtype=torch.int8)
        return torch.cat((d.view(torch.uint8), q.view(torch.uint8)), -1).contiguous()


def _q8_of(w):
    """Weights stored as block_q8_0 bytes (d = amax / 127, q = w / d to nearest)."""
    b = w.reshape(*w.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    q = torch.round(b / d).to(torch.int8)
    return torch.cat((d.half().view(torch.uint8), q.view(torch.uint8)), -1).contiguous()


def _q8_value(blocks):
    """The values of block_q8_0 bytes in 64 bits."""
    d = blocks[..., :2].contiguous().view(torch.float16).double()
    return (blocks[..., 2:].contiguous().view(torch.int8).double() * d).flatten(-2)


def _host(t):
    return t.cpu().numpy()


def _host_q8(blocks):
    return _host(blocks).view(synth.Q8_DTYPE)[..., 0]


def _dac_weights(v, Q, D, N):
    return dict(w_in=v.normal(Q, 8, D, std=D ** -0.5), b_in=v.normal(Q, 8, std=0.1), codebook=v.normal(Q, N, 8),
                w_out=v.normal(Q, D, 8, std=8 ** -0.5), b_out=v.normal(Q, D, std=0.1))


def _dac_stages(w, recipe=aqmi.DAC_FISH):
    return aqmi.DacStages(_context(), *(_host(w[k]) for k in ("w_in", "b_in", "codebook", "w_out", "b_out")), recipe)


def _codes(M, *shape):
    return torch.empty((M,) + shape, dtype=torch.int32, device=DEV)


def _floats(M, *shape, dtype=torch.float32):
    return torch.empty((M,) + shape, dtype=dtype, device=DEV)


def _inputs(case, seed):
    """The weights and inputs of a seed, as torch tensors on the GPU."""
    v, kind = _Values(seed), case["kind"]
    if kind == "decode":
        kind = case["family"] + "_decode"
    if kind == "qwen3":
        S, N, K = case["stages"], case["N"], case["K"]
        usage = v.uniform(1.0, 30.0, S, N)
        return dict(usage=usage, sums=v.normal(S, N, K, std=0.25) * usage[..., None],
                    semantic=v.normal(K, case["T"]), acoustic=v.normal(K, case["T"]))
    if kind == "rvq":
        shape = (case["Q"], case["N"], case["K"])
        std = 1.0 / 16.0 if case["K"] == 256 else 1.0
        x = v.frames(case, case["K"])
        if case["K"] != 256:   # channels of a self-supervised encoder differ in scale
            x = x * v.uniform(0.5, 2.0, case["K"])
        return dict(x=x, codebook=v.q8_blocks(*shape) if case["q8"] else v.normal(*shape, std=std))
    if kind == "rvq_decode":
        return dict(idx=v.codes(case["N"], case["T"], case["Q"]),
                    codebook=v.normal(case["Q"], case["N"], case["K"], std=1.0 / 16.0))
    if kind == "projected":
        Q, N, K, H = case["Q"], case["N"], case["K"], case["H"]
        cb, w_in, w_out = v.normal(Q, N, K), v.normal(Q, K, H, std=H ** -0.5), v.normal(Q, H, K, std=K ** -0.5)
        return dict(x=v.frames(case, H), codebook=_q8_of(cb) if case["cb_q8"] else cb,
                    w_in=_q8_of(w_in) if case["proj_q8"] else w_in, b_in=v.normal(Q, K, std=0.1),
                    w_out=_q8_of(w_out) if case["proj_q8"] else w_out, b_out=v.normal(Q, H, std=0.1))
    if kind in ("fish", "fish_decode"):
        D, N0, N, Q = case["D"], case["N0"], case["N"], case["Q"]
        w = dict(first=_dac_weights(v, 1, D, N0), rest=_dac_weights(v, Q, D, N))
        if kind == "fish":
            return dict(w, x=v.frames(dict(case, channel_major=True), D))
        return dict(w, idx=torch.cat((v.codes(N0, case["T"], 1), v.codes(N, case["T"], Q)), 1).contiguous())
    if kind in ("dac", "outetts"):
        return dict(w=_dac_weights(v, case["Q"], case["D"], case["N"]), x=v.frames(case, case["D"]))
    C, R, N, Q = case["C"], case["R"], case["N"], case["Q"]   # moss, moss_decode

    def conv(*shape):   # a folded weight-normalised 1x1 conv
        u = v.normal(*shape)
        return u * (v.uniform(0.5, 2.0, *shape[:-1], 1) / u.norm(dim=-1, keepdim=True))

    w = dict(input_w=conv(R, C), input_b=v.normal(R, std=0.1), in_w=conv(Q, 8, R), in_b=v.normal(Q, 8, std=0.1),
             codebook=v.normal(Q, N, 8), out_w=conv(Q, R, 8), out_b=v.normal(Q, R, std=0.1), output_w=conv(C, R),
             output_b=v.normal(C, std=0.1))
    return dict(w=w, x=v.normal(case["T"], C)) if kind == "moss" else dict(w=w, idx=v.codes(N, case["T"], Q))


def prepare(case, seed):
    """Uploaded weights, inputs and output buffers of a call."""
    i, kind, ctx = _inputs(case, seed), case["kind"], _context()
    if kind == "decode":
        kind = case["family"] + "_decode"
    M = case.get("B", 1) * case["T"]
    s = dict(kind=kind, M=M, case=case, x=i.get("x"), idx=i.get("idx"))
    if kind == "qwen3":
        es, usage = _host(i["sums"]), _host(i["usage"])
        s.update(semantic=aqmi.Codebooks.from_ema(ctx, es[:1], usage[:1], aqmi.DIRECT),
                 acoustic=aqmi.Codebooks.from_ema(ctx, es[1:], usage[1:], aqmi.DIRECT), xs=i["semantic"],
                 xa=i["acoustic"], idx_s=_codes(M, 1), idx_a=_codes(M, case["stages"] - 1))
    elif kind == "rvq":
        Q, k = case["Q"], case["topk"]
        cbt = aqmi.CB_Q8_0 if case["q8"] else aqmi.CB_F32
        s.update(cb=aqmi.Codebooks.from_device(ctx, i["codebook"], RECIPES[case["recipe"]], cbt,
                                               shape=(Q, case["N"], case["K"])),
                 out=dict(idx=_codes(M, Q), residual=_floats(M, case["K"]) if case["residual"] else None,
                          dist=_floats(M, Q) if case["dist"] else None, topk=k,
                          topk_idx=_codes(M, Q, k) if k else None, topk_dist=_floats(M, Q, k) if k else None))
    elif kind == "rvq_decode":
        s.update(cb=aqmi.Codebooks.from_device(ctx, i["codebook"], aqmi.OMNIVOICE), out=_floats(M, case["K"]))
    elif kind == "projected":
        cb = _host_q8(i["codebook"]) if case["cb_q8"] else _host(i["codebook"])
        w_in, w_out = ((_host_q8 if case["proj_q8"] else _host)(i[k]) for k in ("w_in", "w_out"))
        s.update(cb=aqmi.Codebooks.projected(ctx, cb, w_in, _host(i["b_in"]), w_out, _host(i["b_out"]),
                                             RECIPES[case["recipe"]], aqmi.CB_Q8_0 if case["cb_q8"] else aqmi.CB_F32,
                                             aqmi.CB_Q8_0 if case["proj_q8"] else aqmi.CB_F32),
                 out=dict(idx=_codes(M, case["Q"]), residual=_floats(M, case["H"]) if case["residual"] else None))
    elif kind in ("fish", "fish_decode"):
        s.update(first=_dac_stages(i["first"]), rest=_dac_stages(i["rest"]))
        if kind == "fish":
            s.update(idx=_codes(M, 1 + case["Q"]), residual=_floats(M, case["D"]),
                     recon=_floats(M, case["D"]) if case["recon"] else None)
        else:
            s.update(out=_floats(M, case["D"]))
    elif kind in ("dac", "outetts"):
        s.update(st=_dac_stages(i["w"], aqmi.DAC_OUTETTS if kind == "outetts" else aqmi.DAC_FISH),
                 idx=_codes(M, case["Q"]), residual=_floats(M, case["D"]) if case.get("residual") else None,
                 recon=_floats(M, case["D"]) if case.get("recon") else None)
    else:
        w = i["w"]
        order = ("input_w", "input_b", "in_w", "in_b", "codebook", "out_w", "out_b", "output_w", "output_b")
        s.update(q=aqmi.MossQuantizer(ctx, *(_host(w[k]) for k in order)))
        s.update(idx=_codes(M, case["Q"])) if kind == "moss" else s.update(out=_floats(M, case["C"]))
    return s


# ---- the calls ---------------------------------------------------------------


def run(s):
    kind, M, case = s["kind"], s["M"], s["case"]
    T = case["T"]
    if kind == "qwen3":
        K = case["K"]
        s["semantic"].encode_strided(s["xs"], M, T, K * T, 1, T, s["idx_s"])
        s["acoustic"].encode_strided(s["xa"], M, T, K * T, 1, T, s["idx_a"])
        return dict(semantic=s["idx_s"], acoustic=s["idx_a"])
    if kind in ("rvq", "projected"):
        if case["channel_major"]:
            C = s["x"].shape[1]
            s["cb"].encode_strided(s["x"], M, T, C * T, 1, T, **s["out"])
        else:
            s["cb"].encode(s["x"], **s["out"])
        return {k: v for k, v in s["out"].items() if k != "topk" and v is not None}
    if kind == "rvq_decode":
        s["cb"].decode(s["idx"], s["out"])
        return s["out"]
    if kind == "fish":
        D, ld = case["D"], 1 + case["Q"]
        at = s["idx"].data_ptr()
        s["first"].encode_ex(s["x"], M, T, (D * T, 1, T), at, ld, s["residual"], s["recon"])
        s["rest"].encode_ex(s["residual"], M, T, (D * T, D, 1), at + 4, ld, None, s["recon"], s["recon"] is not None)
        return dict(idx=s["idx"]) if s["recon"] is None else dict(idx=s["idx"], recon=s["recon"])
    if kind == "fish_decode":
        at, ld = s["idx"].data_ptr(), 1 + case["Q"]
        s["first"].decode_ex(at, ld, M, s["out"])
        s["rest"].decode_ex(at + 4, ld, M, s["out"], accumulate=True)
        return s["out"]
    if kind in ("dac", "outetts"):
        if case.get("channel_major"):
            D = case["D"]
            s["st"].encode_ex(s["x"], M, T, (D * T, 1, T), s["idx"].data_ptr(), case["Q"], s["residual"], s["recon"])
        else:
            s["st"].encode(s["x"], T, s["idx"], s["residual"], s["recon"])
        return {k: s[k] for k in ("idx", "residual", "recon") if s[k] is not None}
    if kind == "moss":
        s["q"].encode(s["x"], s["idx"])
        return s["idx"]
    s["q"].decode(s["idx"], s["out"])
    return s["out"]


# ---- what a call cannot do without ------------------------------------------


def work(case):
    """Inputs, weights and outputs once, and the contractions' operations."""
    kind, M = case["kind"], case.get("B", 1) * case["T"]
    if kind == "decode":
        Q = case["Q"] + (1 if case["family"] == "fish" else 0)
        width = {"fish": case.get("D"), "rvq": case.get("K"), "moss": case.get("C")}[case["family"]]
        rows = {"fish": 8 * (case.get("N0", 0) + (Q - 1) * case["N"]) + 9 * width * Q,
                "rvq": Q * case["N"] * (case.get("K") or 0), "moss": Q * case["N"] * 8 + Q * 9 * (case.get("R") or 0)
                + (case.get("R") or 0) * width}[case["family"]]
        per = {"fish": Q * 18 * width, "rvq": Q * width, "moss": Q * width}[case["family"]]
        return dict(bytes=4.0 * (M * (Q + width) + min(rows, M * Q * width)), flops=float(M * per))
    if kind == "qwen3":
        S, N, K = case["stages"], case["N"], case["K"]
        return dict(bytes=4.0 * (2 * M * K + S * N * K + M * S), flops=2.0 * M * S * N * K)
    if kind == "rvq":
        Q, N, K = case["Q"], case["N"], case["K"]
        out = Q * (1 + (1 if case["dist"] else 0) + 2 * case["topk"]) + (K if case["residual"] else 0)
        cb = Q * N * K * (34.0 / 32.0 if case["q8"] else 4.0)
        return dict(bytes=4.0 * M * (K + out) + cb, flops=2.0 * M * Q * N * K)
    if kind == "projected":
        Q, N, K, H = case["Q"], case["N"], case["K"], case["H"]
        weights = Q * N * K * (34.0 / 32.0 if case["cb_q8"] else 4.0) + 2 * Q * K * H * (34.0 / 32.0 if case["proj_q8"] else 4.0)
        return dict(bytes=4.0 * M * (H + Q + (H if case["residual"] else 0)) + weights,
                    flops=2.0 * M * Q * (2 * H * K + N * K))
    if kind in ("dac", "outetts", "fish"):
        D, Q = case["D"], case["Q"] + (1 if kind == "fish" else 0)
        codes = case["Q"] * case["N"] + (case["N0"] if kind == "fish" else 0)
        out = Q + D * ((1 if case.get("recon") else 0) + (1 if case.get("residual") else 0))
        return dict(bytes=4.0 * (M * (D + out) + codes * 8 + Q * 17 * D), flops=M * (16.0 * codes + 33.0 * D * Q))
    C, R, N, Q = case["C"], case["R"], case["N"], case["Q"]
    return dict(bytes=4.0 * (M * (C + Q) + R * C + Q * 17 * R + Q * N * 8),
                flops=M * (2.0 * C * R + Q * (33.0 * R + 16.0 * N)))


# ---- the same in 64 bits -----------------------------------------------------


def _rows(x, case, width):
    """Frames [M, C] in 64 bits."""
    return (x.transpose(1, 2).reshape(-1, width) if x.dim() == 3 else x).double()


def _q8_query(r):
    """The query image of a Q8_0 product: blocks of 32 rounded to 127 steps, fp16 scale."""
    b = r.reshape(r.shape[0], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    q = torch.round(b * torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax)))
    return (q * (amax / 127.0).half().double()).flatten(1)


def _nearest(r, c, q8, k):
    """Codes and squared distances of the k nearest rows of c, best first."""
    e2, codes, dists = (c * c).sum(-1), [], []
    step = max(1, (1 << 27) // c.shape[0])
    for at in range(0, r.shape[0], step):
        p = r[at:at + step]
        d = (p * p).sum(-1, keepdim=True) + e2 - 2.0 * ((_q8_query(p) if q8 else p) @ c.T)
        v, n = d.topk(k, dim=-1, largest=False)
        codes.append(n)
        dists.append(v)
    return torch.cat(codes), torch.cat(dists)


def _exact_rvq(case, i):
    c = _q8_value(i["codebook"]) if case["q8"] else i["codebook"].double()
    r, k = _rows(i["x"], case, case["K"]), case["topk"]
    # the OmniVoice logit 2 c.r - |c|^2 leaves the query's own square out
    shift = case["recipe"] == "omnivoice"
    out = dict(idx=[], dist=[], topk_idx=[], topk_dist=[])
    for q in range(case["Q"]):
        n, d = _nearest(r, c[q], case["q8"], max(1, k))
        if shift:
            d = d - (r * r).sum(-1, keepdim=True)
        out["idx"].append(n[:, 0])
        out["dist"].append(d[:, 0])
        out["topk_idx"].append(n)
        out["topk_dist"].append(d)
        r = r - c[q][n[:, 0]]
    out = {name: torch.stack(v, 1) for name, v in out.items()}
    got = dict(idx=out["idx"].int())
    if case["residual"]:
        got["residual"] = r
    if case["dist"]:
        got["dist"] = out["dist"]
    if k:
        got.update(topk_idx=out["topk_idx"].int(), topk_dist=out["topk_dist"])
    return got


def _exact_projected(case, i):
    value = lambda t, q8: _q8_value(t) if q8 else t.double()  # noqa: E731
    c, w_in, w_out = value(i["codebook"], case["cb_q8"]), value(i["w_in"], case["proj_q8"]), value(i["w_out"], case["proj_q8"])
    r, codes = _rows(i["x"], case, case["H"]), []
    quant = _q8_query if case["proj_q8"] else (lambda t: t)
    for q in range(case["Q"]):
        p = quant(r) @ w_in[q].T + i["b_in"][q].double()
        n = _nearest(p, c[q], case["cb_q8"], 1)[0][:, 0]
        r = r - (quant(c[q])[n] @ w_out[q].T + i["b_out"][q].double())
        codes.append(n)
    got = dict(idx=torch.stack(codes, 1).int())
    if case["residual"]:
        got["residual"] = r
    return got


def _exact_dac(w, r, recon, codes, eps=1e-12):
    """The stages of w on the residual r; codes are appended."""
    for q in range(w["w_in"].shape[0]):
        c = w["codebook"][q].double()
        p = r @ w["w_in"][q].double().T + w["b_in"][q].double()
        p = p / (p * p).sum(-1, keepdim=True).add(eps).sqrt()
        n = (p @ torch.nn.functional.normalize(c, dim=-1).T).argmax(-1)
        z = c[n] @ w["w_out"][q].double().T + w["b_out"][q].double()
        r, recon = r - z, recon + z
        codes.append(n)
    return r, recon


def exact(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    if kind == "decode":
        kind = case["family"] + "_decode"
    if kind == "qwen3":
        c = i["sums"].double() / i["usage"].double()[..., None]
        got = []
        for x, books in ((i["semantic"], c[:1]), (i["acoustic"], c[1:])):
            r, codes = x.T.double(), []
            for book in books:
                codes.append(_nearest(r, book, False, 1)[0][:, 0])
                r = r - book[codes[-1]]
            got.append(torch.stack(codes, 1).int())
        return dict(semantic=got[0], acoustic=got[1])
    if kind == "rvq":
        return _exact_rvq(case, i)
    if kind == "projected":
        return _exact_projected(case, i)
    if kind == "rvq_decode":
        c, idx = i["codebook"].double(), i["idx"].long()
        return sum(c[q][idx[:, q]] for q in range(case["Q"]))
    if kind == "fish":
        r, codes = _rows(i["x"], case, case["D"]), []
        recon = torch.zeros_like(r)
        for w in (i["first"], i["rest"]):
            r, recon = _exact_dac(w, r, recon, codes)
        got = dict(idx=torch.stack(codes, 1).int())
        return dict(got, recon=recon) if case["recon"] else got
    if kind == "fish_decode":
        idx, z = i["idx"].long(), 0.0
        stages = [(i["first"], 0)] + [(i["rest"], q) for q in range(case["Q"])]
        for s, (w, q) in enumerate(stages):
            z = z + w["codebook"][q].double()[idx[:, s]] @ w["w_out"][q].double().T + w["b_out"][q].double()
        return z
    if kind in ("dac", "outetts"):
        r, codes = _rows(i["x"], case, case["D"]), []
        r, recon = _exact_dac(i["w"], r, torch.zeros_like(r), codes, 0.0 if kind == "outetts" else 1e-12)
        got = dict(idx=torch.stack(codes, 1).int())
        if case.get("residual"):
            got["residual"] = r
        return dict(got, recon=recon) if case.get("recon") else got
    w = {k: t.double() for k, t in i["w"].items()}
    if kind == "moss_decode":
        z = w["out_b"].sum(0) + sum(w["codebook"][q][i["idx"][:, q].long()] @ w["out_w"][q].T for q in range(case["Q"]))
        return z @ w["output_w"].T + w["output_b"]
    r, codes = i["x"].double() @ w["input_w"].T + w["input_b"], []
    for q in range(case["Q"]):
        e = torch.nn.functional.normalize(r @ w["in_w"][q].T + w["in_b"][q], dim=-1)
        n = (e @ torch.nn.functional.normalize(w["codebook"][q], dim=-1).T).argmax(-1)
        r = r - (w["codebook"][q][n] @ w["out_w"][q].T + w["out_b"][q])
        codes.append(n)
    return torch.stack(codes, 1).int()
