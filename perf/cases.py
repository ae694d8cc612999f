"""Performance cases of the framework: the calls that a text-to-audio program makes, as it makes them.

One generation encodes the prompt (two text encoders), prepares the conditioning, evaluates the DiT
at every sampler step and decodes the latent to audio; a program that composes its own graph calls the
runtime's launchers. Device memory is torch's: the library takes device pointers, so a torch tensor's
storage serves as input or output of any call.

Weights are random with the scales of the package's synthetic generators, drawn once per shape from a
fixed seed (a program keeps one set); inputs are drawn from the case's seed.
"""
import ctypes
import importlib
import math

import numpy as np
import torch

tsn = importlib.import_module("thinksound-native_amd")

DEV = "cuda"
WEIGHT_SEED = 4242
F64 = torch.float64


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the timestep MLP and global vector of a program that composes its graph from launchers: five
        # launches on one row, latency only
        {"name": "time_mlp", "kind": "tmlp", "H": 1024, "K": 256, "wdt": "bf16"},
        # launcher GEMM of a text stream's FFN (154 rows, f32 activations, f16 weights)
        {"name": "gemm_154x2816x1024", "kind": "gemm", "M": 154, "N": 2816, "K": 1024, "xdt": "f32", "bias": False},
        # launcher attention of one sample's joint rows, a ragged length (f32 in and out)
        {"name": "attention_331", "kind": "attention", "S": 331, "nh": 16},
        # one joint block of the 30 s clip under CFG (two samples)
        {"name": "joint_block_30s", "kind": "block", "joint": True, "B": 2, "La": 960, "Lt": 141, "H": 1024, "conv": True},
        # one fused block of the throughput batch: eight prompts under CFG
        {"name": "fused_block_b16", "kind": "block", "joint": False, "B": 16, "La": 256, "Lt": 141, "H": 1024, "conv": True},
        # a whole velocity evaluation of the 8 s clip under CFG, replayed as a graph
        {"name": "dit_eval_8s", "kind": "dit", "B": 2, "La": 256, "Lt": 141, "n_joint": 7, "n_fused": 14, "graph": True},
        # a whole velocity evaluation of the checkpoint's three-stream graph, 8 s under CFG, eager
        {"name": "ref_eval_8s", "kind": "ref", "B": 2, "T": 172, "C": 64, "TS": 154, "n_joint": 7, "n_fused": 14},
        # conditioning prep of one 8 s generation: video streams once, then both CFG text arms
        {"name": "cond_8s", "kind": "cond", "T": 172, "C": 64, "sync_S": 192, "TS": 154},
        # the pooled-text encoder on one prompt
        {"name": "clip_encode", "kind": "clip", "H": 1024, "NL": 24, "ctx": 77},
        # the token-text encoder on one prompt
        {"name": "t5_encode", "kind": "t5", "d": 2048, "d_ff": 5120, "NL": 24, "ctx": 77},
        # decoding a one-second latent (a preview, or the tail segment of a longer clip)
        {"name": "vae_1s", "kind": "vae", "T": 22},
        # decoding the 8 s latent
        {"name": "vae_8s", "kind": "vae", "T": 172},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tmlp", "gemm", "attention", "block", "block", "block", "dit", "ref", "ref", "cond", "clip", "t5", "vae", "vae"])
    if kind == "tmlp":   # other widths, odd ones among them, and every weight type
        return {"kind": kind, "H": 8 * _log_int(rng, 32, 256), "K": 8 * _log_int(rng, 16, 256),
                "wdt": rng.choice(["bf16", "f16", "f32"])}
    if kind == "gemm":   # a launcher GEMM of one stream: 16 rows to the 30 s clip's two samples
        return {"kind": kind, "M": _log_int(rng, 16, 2202), "N": 8 * _log_int(rng, 32, 512),
                "K": 64 * _log_int(rng, 4, 64), "xdt": rng.choice(["f32", "f32", "f16"]), "bias": rng.random() < 0.5}
    if kind == "attention":
        return {"kind": kind, "S": _log_int(rng, 32, 1101), "nh": rng.choice([8, 12, 16])}
    if kind == "block":   # clips of 1 s to 30 s, batches up to 8 prompts under CFG
        B = rng.choice([1, 2, 2, 4, 8, 16])
        La = _log_int(rng, 32, min(960, 4096 // B))
        return {"kind": kind, "joint": rng.random() < 0.5, "B": B, "La": La, "Lt": rng.randint(20, 141),
                "H": rng.choice([512, 1024, 1024, 1024]), "conv": rng.random() < 0.75}
    if kind == "dit":
        return {"kind": kind, "B": 2, "La": _log_int(rng, 32, 256), "Lt": rng.randint(20, 141),
                "n_joint": rng.randint(1, 7), "n_fused": rng.randint(0, 14), "graph": rng.random() < 0.5}
    if kind == "ref":   # clips of 1 s to 8 s
        d = rng.uniform(1.0, 8.0)
        return {"kind": kind, "B": rng.choice([1, 2, 2]), "T": int(round(44100.0 / 2048.0 * d)), "C": max(1, int(8 * d)),
                "TS": rng.choice([77, 131, 154]), "n_joint": rng.randint(1, 7), "n_fused": rng.randint(0, 14)}
    if kind == "cond":
        d = rng.uniform(1.0, 8.0)
        return {"kind": kind, "T": int(round(44100.0 / 2048.0 * d)), "C": max(1, int(8 * d)),
                "sync_S": max(8, int(24 * d)), "TS": rng.choice([77, 131, 154])}
    if kind == "clip":
        return {"kind": kind, "H": rng.choice([512, 768, 1024]), "NL": rng.randint(2, 24), "ctx": rng.randint(8, 77)}
    if kind == "t5":
        d = rng.choice([512, 768, 1024, 2048])
        return {"kind": kind, "d": d, "d_ff": {512: 1024, 768: 2048, 1024: 2816, 2048: 5120}[d],
                "NL": rng.randint(2, 24 if d < 2048 else 20), "ctx": rng.randint(8, 77)}
    return {"kind": "vae", "T": _log_int(rng, 5, 172)}


# ---------------------------------------------------------------- handles

class Dev:
    """A torch tensor as the library's calls take a device array: pointer, size, shape."""

    def __init__(self, t):
        self.t = t
        self.p = ctypes.c_void_p(t.data_ptr())
        self.nbytes = t.numel() * t.element_size()
        self.shape = tuple(t.shape)


class Handle:
    """A loaded model on the program's runtime; closed when the last state drops it."""

    def __init__(self, model):
        self.model = model

    def __del__(self):
        self.model.close()


_last = {"weights": (None, None), "handle": (None, None), "runtime": (None, None)}


def _kept(what, key, make):
    """make() for `key`, kept until another key is asked for."""
    if _last[what][0] != key:
        _last[what] = (None, None)
        _last[what] = (key, make())
    return _last[what][1]


def _dit_spec(case):
    if case["kind"] == "block":
        j = 1 if case["joint"] else 0
        return tsn.default_spec(1).copy(B=case["B"], La=case["La"], Lt=case["Lt"], H=case["H"], NH=case["H"] // 64,
                                        F=4 * case["H"], n_joint=j, n_fused=1 - j, audio_ffn_conv=int(case["conv"]))
    return tsn.default_spec(1).copy(B=case["B"], La=case["La"], Lt=case["Lt"], n_joint=case["n_joint"],
                                    n_fused=case["n_fused"])


def _spec(case):
    k = case["kind"]
    if k in ("block", "dit"):
        return _dit_spec(case)
    if k == "ref":
        return tsn.ref_spec_for_duration(8, case["B"]).copy(T=case["T"], C=case["C"], TS=case["TS"],
                                                            n_joint=case["n_joint"], n_fused=case["n_fused"])
    if k == "cond":
        return tsn.cond_spec_for_duration(8).copy(T=case["T"], C=case["C"], sync_S=case["sync_S"], TS=case["TS"])
    if k == "clip":
        return tsn.clip_spec_default().copy(H=case["H"], NH=case["H"] // 64, NL=case["NL"], ctx=case["ctx"])
    if k == "t5":
        return tsn.t5_spec_default().copy(d=case["d"], NH=case["d"] // 64, d_ff=case["d_ff"], NL=case["NL"], ctx=case["ctx"])
    return tsn.vae_spec_for_duration(8).copy(T=case["T"])


_MANIFEST = {"block": "manifest", "dit": "manifest", "ref": "ref_manifest", "cond": "cond_manifest",
             "clip": "clip_manifest", "t5": "t5_manifest", "vae": "vae_manifest"}
_MODEL = {"block": "DitModel", "dit": "DitModel", "ref": "RefDitModel", "cond": "RefCondModel", "clip": "ClipModel",
          "t5": "T5Model", "vae": "VaeModel"}


def _manifest(case):
    return getattr(tsn, _MANIFEST[case["kind"]])(_spec(case))


def _scale(kind, name, numel, spec):
    """(mean, std) of one weight tensor, as the package's synthetic generators choose them."""
    if kind in ("block", "dit", "ref", "cond"):
        return (1.0 if name.endswith("norm.weight") else 0.0), 0.02
    if kind == "vae":
        if name.endswith((".alpha", ".beta")):
            return 0.0, 0.1
        if name.endswith(".bias"):
            return 0.0, 0.02
        layer = int(name.split(".")[2])
        oc = spec.width[0] if layer == 0 else spec.out_ch if layer == 7 else spec.width[layer]
        return 0.0, (0.5 if name.endswith(".layers.3.weight") and layer != 7 else 1.0) / math.sqrt(numel / oc)
    if name in ("tok_emb", "pos_emb"):
        return 0.0, 1.0
    if name == "rel_bias":
        return 0.0, 0.5
    if name.endswith(("norm", "ln1.w", "ln2.w", "out_ln.w")):
        return 1.0, 0.1
    if name.endswith(".b"):
        return 0.0, 0.02
    fan = spec.d_ff if name.endswith(".wo") else 4 * spec.H if name.endswith(".fc2.w") else spec.d if kind == "t5" else spec.H
    gain = 0.5 if name.endswith((".out.w", ".fc2.w", ".o", ".wo")) else 1.0
    if kind == "t5" and name.endswith(".q"):
        gain = 0.125   # the checkpoints fold 1/sqrt(64) into q
    return 0.0, gain / math.sqrt(fan)


def _weights(case):
    """The flat host weight buffer that the model uploads: bf16 bits, or f32 for the f32 models."""
    spec, kind = _spec(case), case["kind"]
    key = (kind if kind != "block" else "dit", tuple(sorted((k, str(v)) for k, v in spec.as_dict().items())))

    def make():
        man = _manifest(case)
        g = torch.Generator(DEV).manual_seed(WEIGHT_SEED)
        bf16 = kind in ("block", "dit", "ref", "cond")
        flat = torch.empty(man[-1][2] + man[-1][1], device=DEV, dtype=torch.bfloat16 if bf16 else torch.float32)
        for name, numel, off in man:
            mean, std = _scale(kind, name, numel, spec)
            flat[off:off + numel] = torch.randn(numel, device=DEV, generator=g) * std + mean
        host = (flat.view(torch.int16) if bf16 else flat).cpu().numpy()
        return host.view(np.uint16) if bf16 else host

    return key, _kept("weights", key, make)


def _runtime():
    """The program's one runtime: one GPU, one stream."""
    return _kept("runtime", 0, lambda: tsn.Runtime(0))


def _handle(case, own=False):
    """The case's loaded model (None for launcher cases). A captured graph belongs to its model, so a
    state that keeps a graph has a model of its own."""
    if case["kind"] not in _MODEL:
        return None
    key, w = _weights(case)

    def make():
        m = getattr(tsn, _MODEL[case["kind"]])(_runtime(), _spec(case))
        m.upload_weights(w)
        return Handle(m)

    return make() if own else _kept("handle", key, make)


# ---------------------------------------------------------------- inputs

def _inputs(case, seed):
    """Every input of the case as torch tensors on the GPU (token ids: host arrays), from the seed alone."""
    g = torch.Generator(DEV).manual_seed(1000003 * int(seed) + 17)

    def rn(*shape, std=1.0):
        return torch.randn(*shape, device=DEV, generator=g) * std

    k = case["kind"]
    if k == "tmlp":   # a sinusoid's values, and the pooled features that the embedding is added to
        dt, H, K = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[case["wdt"]], case["H"], case["K"]
        return {"W0": rn(H, K, std=0.02).to(dt), "b0": rn(H, std=0.02), "W2": rn(H, H, std=0.02).to(dt),
                "b2": rn(H, std=0.02), "x": (rn(K) * 100.0).cos(), "pooled": rn(H)}
    if k == "gemm":
        return {"W": rn(case["N"], case["K"], std=0.02).half(), "b": rn(case["N"], std=0.02) if case["bias"] else None,
                "X": rn(case["M"], case["K"]).to(torch.float16 if case["xdt"] == "f16" else torch.float32)}
    if k == "attention":   # q and k after a per-head RMS norm, as the DiT's launcher graph passes them
        S, nh = case["S"], case["nh"]
        qkv = rn(S, 3, nh, 64)
        qkv[:, :2] /= qkv[:, :2].square().mean(-1, keepdim=True).sqrt()
        return {"qkv": qkv.reshape(S, 3 * nh * 64).contiguous()}
    s = _spec(case)
    if k == "block":
        return {"X": rn(s.B, s.La + s.Lt, s.H), "g": rn(s.B, s.H)}
    if k == "dit":   # (cond, uncond) pairs: shared latent and time, zero text features on the second arm
        z, text, pooled = rn(1, s.La, s.latent), torch.zeros(2, s.Lt, s.H, device=DEV), torch.zeros(2, s.H, device=DEV)
        text[0], pooled[0] = rn(s.Lt, s.H), rn(s.H)
        t = torch.rand(1, device=DEV, generator=g)
        return {"z": z.repeat(2, 1, 1), "t": t.repeat(2), "text": text, "pooled": pooled}
    if k == "ref":
        x, clip, sync = rn(1, s.T, s.latent), rn(1, s.C, s.H), rn(1, s.T, s.H)
        t = torch.rand(1, device=DEV, generator=g)
        return {"x": x.repeat(s.B, 1, 1), "t": t.repeat(s.B), "clip": clip.repeat(s.B, 1, 1), "sync": sync.repeat(s.B, 1, 1),
                "text": rn(s.B, s.TS, s.H), "gcmlp": rn(s.B, s.H)}
    if k == "cond":
        return {"clip_f": rn(s.C, s.clip_dim), "sync_f": rn(s.sync_S, s.sync_dim),
                "text_cat": rn(2, s.TS, s.text_dim), "gtext": rn(2, s.gtext_dim)}
    if k in ("clip", "t5"):   # a prompt of a third of the context or more, then end and padding ids
        r = np.random.default_rng(int(seed))
        n = int(r.integers(max(2, s.ctx // 3), s.ctx + 1))
        ids = np.zeros(s.ctx, np.int32)
        ids[:n] = r.integers(2, s.vocab - 2, n)
        ids[n - 1] = s.vocab - 1 if k == "clip" else 1
        return {"ids": ids}
    return {"latent": rn(s.T, s.latent)}


def _outputs(case):
    k = case["kind"]
    if k == "tmlp":
        return {"h": (case["H"],), "emb": (case["H"],), "g": (case["H"],)}
    if k == "gemm":
        return {"y": (case["M"], case["N"])}
    if k == "attention":
        return {"y": (case["S"], case["nh"] * 64)}
    s = _spec(case)
    if k == "block":
        return {"X": (s.B, s.La + s.Lt, s.H)}
    if k == "dit":
        return {"v": (s.B, s.La, s.latent)}
    if k == "ref":
        return {"flow": (s.B, s.T, s.latent)}
    if k == "cond":
        return {"clip_pp": (s.C, s.H), "sync_gather": (s.T, s.H), "clip_fc": (s.H,), "text_pp0": (s.TS, s.H),
                "gcmlp0": (s.H,), "text_pp1": (s.TS, s.H), "gcmlp1": (s.H,)}
    if k == "clip":
        return {"per_token": (s.ctx, s.H), "pooled": (s.H,)}
    if k == "t5":
        return {"per_token": (s.ctx, s.d)}
    return {"audio": (tsn.vae_audio_len(s), s.out_ch)}


class State:
    """What a program holds before the call: the handle, its inputs and the output buffers."""

    def __init__(self, case, seed):
        self.case = case
        self.inp = _inputs(case, seed)
        self.out = {n: torch.empty(shape, device=DEV) for n, shape in _outputs(case).items()}
        self.i = {n: Dev(t) if isinstance(t, torch.Tensor) else t for n, t in self.inp.items()}
        self.o = {n: Dev(t) for n, t in self.out.items()}
        graph = case["kind"] == "dit" and case["graph"]
        self.h, self.rt = _handle(case, own=graph), _runtime()
        self.m = self.h.model if self.h is not None else None
        if case["kind"] == "cond":   # each text arm's rows of the stacked inputs
            self.arm = [(Dev(self.inp["text_cat"][a]), Dev(self.inp["gtext"][a])) for a in range(2)]
        if graph:
            torch.cuda.synchronize()   # the capture runs on the library's own stream
            self.m.capture_forward(self.i["z"], self.i["t"], self.i["text"], self.i["pooled"], self.o["v"])


def prepare(case, seed):
    return State(case, seed)


_DT = {"f32": tsn.F32, "f16": tsn.F16, "bf16": tsn.BF16}


def run(st):
    c, i, o, m, rt = st.case, st.i, st.o, st.m, st.rt
    k = c["kind"]
    if k == "tmlp":
        H, K, dt = c["H"], c["K"], _DT[c["wdt"]]
        rt.gemv(i["W0"], dt, i["x"], o["h"], i["b0"], H, K)
        rt.silu(o["h"], H)
        rt.gemv(i["W2"], dt, o["h"], o["emb"], i["b2"], H, H)
        rt.add_(i["pooled"], o["emb"], o["g"], H)
        rt.silu(o["g"], H)
    elif k == "gemm":
        rt.gemm(tsn.F16, i["W"], i["X"], _DT[c["xdt"]], o["y"], tsn.F32, i["b"], c["M"], c["N"], c["K"])
    elif k == "attention":
        w = c["nh"] * 64
        rt.attention(i["qkv"], o["y"], c["S"], c["nh"], 64, 3 * w, w, 0, w, 2 * w, 0, 0.125)
    elif k == "block":   # the block updates the residual stream in place
        rt.copy(i["X"], o["X"], st.out["X"].numel())
        (m.joint_block if c["joint"] else m.fused_block)(0, o["X"], i["g"])
    elif k == "dit":
        if c["graph"]:
            m.replay()
        else:
            m.forward_ex(i["z"], i["t"], i["text"], i["pooled"], o["v"])
    elif k == "ref":
        m.forward_ex(i["x"], i["t"], i["clip"], i["text"], i["gcmlp"], i["sync"], o["flow"])
    elif k == "cond":
        m.prep_conditioning(i["clip_f"], i["sync_f"], o["clip_pp"], o["sync_gather"], o["clip_fc"])
        for a, (text_cat, gtext) in enumerate(st.arm):
            m.prep_text_arm(text_cat, gtext, o["clip_fc"], o["text_pp%d" % a], o["gcmlp%d" % a])
    elif k == "clip":
        m.encode(i["ids"], o["per_token"], o["pooled"])
    elif k == "t5":
        m.encode(i["ids"], o["per_token"])
    else:
        m.decode(i["latent"], o["audio"])
    return st.out


# ---------------------------------------------------------------- work

def work(case):
    k = case["kind"]
    out_bytes = 4 * sum(int(np.prod(s)) for s in _outputs(case).values())
    if k == "tmlp":
        H, kk = case["H"], case["K"]
        return {"bytes": H * (kk + H) * (4 if case["wdt"] == "f32" else 2) + 4 * (kk + 3 * H) + out_bytes,
                "flops": 2.0 * H * (kk + H)}
    if k == "gemm":
        m, n, kk = case["M"], case["N"], case["K"]
        return {"bytes": 2 * n * kk + m * kk * (2 if case["xdt"] == "f16" else 4) + (4 * n if case["bias"] else 0) + out_bytes,
                "flops": 2.0 * m * n * kk}
    if k == "attention":
        s, nh = case["S"], case["nh"]
        return {"bytes": 4 * s * 3 * nh * 64 + out_bytes, "flops": 4.0 * s * s * nh * 64}
    s = _spec(case)
    man = _manifest(case)
    wsize = 4 if k in ("clip", "t5", "vae") else 2
    wts = sum(n for name, n, _ in man if name != "tok_emb")
    if k in ("block", "dit"):
        H, F, B, S, nj, nf = s.H, s.F, s.B, s.La + s.Lt, s.n_joint, s.n_fused
        ta = 3 if s.audio_ffn_conv else 1
        att = 4.0 * B * S * S * H
        joint = 8.0 * B * S * H * H + 4.0 * B * H * F * (ta * s.La + s.Lt) + att + 24.0 * B * H * H
        fused = 8.0 * B * S * H * H + 4.0 * B * S * H * F + att + 12.0 * B * H * H
        if k == "block":   # the block's own weights, the stream and g
            pre = "joint_blocks." if case["joint"] else "fused_blocks."
            wts = sum(n for name, n, _ in man if name.startswith(pre))
            return {"bytes": 2 * wts + 4 * (B * S * H + B * H) + out_bytes, "flops": joint if case["joint"] else fused}
        ends = B * (2.0 * H * (s.temb_dim + H) + 4.0 * H * H) + 4.0 * B * s.La * s.latent * H
        return {"bytes": 2 * wts + 4 * B * (s.La * s.latent + s.Lt * H + H + 1) + out_bytes,
                "flops": nj * joint + nf * fused + ends}
    if k == "ref":
        H, F, B, T, C, TS, nj, nf = s.H, s.F, s.B, s.T, s.C, s.TS, s.n_joint, s.n_fused
        S = T + C + TS

        def stream(rows, taps, post=True):   # QKV, then out-proj and SwiGLU FFN
            return 6.0 * rows * H * H + (taps * (2.0 * rows * H * H + 6.0 * rows * H * F) if post else 0.0)

        fl = 0.0
        for j in range(nj):
            post = j < nj - 1
            fl += stream(T, 3) + stream(C, 3, post) + stream(TS, 1, post) + 4.0 * S * S * H
            fl += 12.0 * T * H * H + 2 * (12.0 if post else 4.0) * H * H
        fl += nf * (stream(T, 3) + 4.0 * T * T * H + 12.0 * T * H * H)
        fl += 6.0 * T * s.latent * H + 18.0 * T * H * F + 4.0 * H * H + 4.0 * T * H * H + 14.0 * T * H * s.latent
        return {"bytes": 2 * wts + 4 * B * (T * s.latent + (T + C + TS + 1) * H + 1) + out_bytes, "flops": B * fl}
    if k == "cond":
        H, F = s.H, s.F
        fl = s.sync_S * (14.0 * s.sync_dim * H + 18.0 * H * F) + s.C * (2.0 * s.clip_dim * H + 18.0 * H * F) + 2.0 * H * H
        fl += 2 * (s.TS * (2.0 * s.text_dim * H + 6.0 * H * F) + 2.0 * s.gtext_dim * H + 6.0 * H * F)
        ins = s.C * s.clip_dim + s.sync_S * s.sync_dim + 2 * (s.TS * s.text_dim + s.gtext_dim)
        return {"bytes": 2 * wts + 4 * ins + out_bytes, "flops": fl}
    if k == "clip":
        n, H = s.ctx, s.H
        return {"bytes": wsize * (wts + n * H) + 4 * n + out_bytes,
                "flops": s.NL * (24.0 * n * H * H + 4.0 * n * n * H) + 2.0 * H * H}
    if k == "t5":
        n, d = s.ctx, s.d
        return {"bytes": wsize * (wts + n * d) + 4 * n + out_bytes,
                "flops": s.NL * (8.0 * n * d * d + 6.0 * n * d * s.d_ff + 4.0 * n * n * d)}
    T, fl = s.T, 2.0 * s.T * s.width[0] * s.latent * 7
    for n in range(5):
        ci, co = s.width[n], s.width[n + 1]
        T *= s.stride[n]
        fl += 2.0 * T * ci * co * (s.kt[n] // s.stride[n]) + 3 * 16.0 * T * co * co
    return {"bytes": wsize * wts + 4 * s.T * s.latent + out_bytes, "flops": fl + 14.0 * T * s.width[5] * s.out_ch}


def tolerance(case):
    """About four times what the start was measured to differ from exact() by: the worst output of
    the listed and drawn cases of the kind is beside each line."""
    k = case["kind"]
    if k in ("tmlp", "gemm"):
        return {"rel": 1e-6}           # f32-accurate products and 32-bit sums: 1.7e-7
    if k == "attention":
        return {"rel": 1.6e-3}         # q, k, v and the probabilities in f16: 4.1e-4
    if k == "block":
        return {"rel": 7e-4}           # f16 operands, f32 residual stream: 1.7e-4
    if k in ("dit", "ref"):
        return {"rel": 1.5e-3}         # the same through up to 21 blocks: 3.7e-4
    if k == "cond":
        return {"rel": 4e-5}           # f32-accurate operands: 9.1e-6
    if k in ("clip", "t5"):
        return {"rel": 5e-6}           # f32 products and sums through up to 24 layers: 1.1e-6
    return {"rel": 2e-5}               # f32-accurate convs through the decoder: 4.4e-6


# ---------------------------------------------------------------- 64-bit results

class _Named:
    """The case's weights by name, in 64 bits on the GPU, converted when asked for."""

    def __init__(self, case):
        _, w = _weights(case)
        t = torch.from_numpy(w.view(np.int16) if w.dtype == np.uint16 else w).to(DEV)
        self.flat = t.view(torch.bfloat16) if w.dtype == np.uint16 else t
        self.at = {n: (off, numel) for n, numel, off in _manifest(case)}

    def __call__(self, name, *shape):
        off, n = self.at[name]
        t = self.flat[off:off + n].to(F64)
        return t.reshape(shape) if shape else t


def _conv(x, w, b=None, dil=1):
    """Same-length conv over rows: x [T, IC], w [OC, IC, K]."""
    K = w.shape[2]
    pad = (K - 1) // 2 * dil
    xp = torch.nn.functional.pad(x, (0, 0, pad, pad))
    y = sum(xp[k * dil:k * dil + x.shape[0]] @ w[:, :, k].t() for k in range(K))
    return y if b is None else y + b


def _ln(x, shift, scale, eps):
    c = x - x.mean(-1, keepdim=True)
    return c / (c.square().mean(-1, keepdim=True) + eps).sqrt() * (1.0 + scale) + shift


def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _rope(x, fscale, theta):
    """x [rows, nh, 64], pairs (2j, 2j+1) turned by row * fscale * theta^(-2j/64)."""
    n = x.shape[0]
    ang = torch.arange(n, device=DEV, dtype=F64)[:, None] * fscale * theta ** (-torch.arange(32, device=DEV, dtype=F64) / 32.0)
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(x.shape)


def _attend(q, k, v, scale, bias=None):
    """q, k, v [S, nh, 64] -> [S, nh * 64]; bias [nh, S, S] is added to the scores."""
    q, k, v = (t.permute(1, 0, 2).contiguous() for t in (q, k, v))
    s = q @ k.transpose(1, 2).contiguous() * scale
    if bias is not None:
        s = s + bias
    return (s.softmax(-1) @ v).permute(1, 0, 2).reshape(q.shape[1], -1)


def _silu(x):
    return x * torch.sigmoid(x)


def _sinusoid(t, dim, max_period):
    f = 10000.0 / max_period * 10000.0 ** (-2.0 * torch.arange(dim // 2, device=DEV, dtype=F64) / dim)
    # the angle reaches 10^4 radians and is defined by its f32 value: t * f rounded to 32 bits
    a = (t.float() * f.float()).to(F64)
    return torch.cat([a.cos(), a.sin()])


def _stream_qkv(W, p, s, x, mod, fscale, interleaved):
    H = s.H
    qkv = _ln(x, mod[0], mod[1], s.ln_eps) @ W(p + ".attn.qkv.weight", 3 * H, H).t() + W(p + ".attn.qkv.bias")
    q, k, v = (qkv[:, j::3] for j in range(3)) if interleaved else qkv.split(H, 1)
    q, k, v = (t.reshape(x.shape[0], s.NH, 64) for t in (q, k, v))
    q, k = _rms(q, W(p + ".attn.q_norm.weight"), s.rms_eps), _rms(k, W(p + ".attn.k_norm.weight"), s.rms_eps)
    if fscale is not None:
        rows = fscale[1]
        q, k = (torch.cat([_rope(t[:rows], fscale[0], s.rope_theta), t[rows:]]) for t in (q, k))
    return q, k, v


def _dit_post(W, p, s, x, att, mod, conv):
    H, F = s.H, s.F
    x = x + mod[2] * (att @ W(p + ".linear1.weight", H, H).t() + W(p + ".linear1.bias"))
    xn = _ln(x, mod[3], mod[4], s.ln_eps)
    if conv:
        return x + mod[5] * _conv(_silu(_conv(xn, W(p + ".ffn.w1.weight", F, H, 3))), W(p + ".ffn.w2.weight", H, F, 3))
    return x + mod[5] * (_silu(xn @ W(p + ".ffn.w1.weight", F, H).t()) @ W(p + ".ffn.w2.weight", H, F).t())


def _mod(W, p, gs, chunks, H):
    """adaLN rows: gs [H] or [rows, H] -> `chunks` tensors of the same leading shape."""
    return (gs @ W(p + ".adaLN_modulation.1.weight", chunks * H, H).t() + W(p + ".adaLN_modulation.1.bias")).split(H, -1)


def _dit_joint(W, i, s, X, gs):
    p = ["joint_blocks.%d.%s" % (i, n) for n in ("latent_block", "text_block")]
    xs = X.split([s.La, s.Lt])
    mods = [_mod(W, n, gs, 6, s.H) for n in p]
    q, k, v = (torch.cat(t) for t in zip(*(_stream_qkv(W, p[j], s, xs[j], mods[j], (1.0, s.La) if j == 0 else None, False)
                                           for j in range(2))))
    att = _attend(q, k, v, 0.125).split([s.La, s.Lt])
    return torch.cat([_dit_post(W, p[j], s, xs[j], att[j], mods[j], j == 0 and s.audio_ffn_conv) for j in range(2)])


def _dit_fused(W, i, s, X, gs):
    p = "fused_blocks.%d" % i
    mod = _mod(W, p, gs, 6, s.H)
    return _dit_post(W, p, s, X, _attend(*_stream_qkv(W, p, s, X, mod, (1.0, s.La), False), 0.125), mod, False)


def _exact_dit(case, inp):
    s, W = _spec(case), _Named(case)
    H, out = s.H, []
    for b in range(s.B):
        if case["kind"] == "block":
            f = _dit_joint if case["joint"] else _dit_fused
            out.append(f(W, 0, s, inp["X"][b].to(F64), _silu(inp["g"][b].to(F64))))
            continue
        te = _sinusoid(inp["t"][b], s.temb_dim, s.t_max_period) @ W("t_embed.mlp.0.weight", H, s.temb_dim).t() + W("t_embed.mlp.0.bias")
        g = _silu(te) @ W("t_embed.mlp.2.weight", H, H).t() + W("t_embed.mlp.2.bias") + inp["pooled"][b].to(F64)
        gs = _silu(g)
        a = inp["z"][b].to(F64) @ W("audio_input_proj.weight", H, s.latent).t() + W("audio_input_proj.bias")
        X = torch.cat([a, inp["text"][b].to(F64)])
        for i in range(s.n_joint):
            X = _dit_joint(W, i, s, X, gs)
        for i in range(s.n_fused):
            X = _dit_fused(W, i, s, X, gs)
        m = _mod(W, "final_layer", gs, 2, H)
        out.append(_ln(X[:s.La], m[0], m[1], s.ln_eps) @ W("final_layer.linear.weight", s.latent, H).t() + W("final_layer.linear.bias"))
    return {"X" if case["kind"] == "block" else "v": torch.stack(out)}


def _swiglu(W, p, x, H, F, conv):
    if conv:
        h = _silu(_conv(x, W(p + ".w1.weight", F, H, 3))) * _conv(x, W(p + ".w3.weight", F, H, 3))
        return _conv(h, W(p + ".w2.weight", H, F, 3))
    h = _silu(x @ W(p + ".w1.weight", F, H).t()) * (x @ W(p + ".w3.weight", F, H).t())
    return h @ W(p + ".w2.weight", H, F).t()


def _ref_post(W, p, s, x, att, mod, conv):
    H = s.H
    b = W(p + ".linear1.bias")
    o = _conv(att, W(p + ".linear1.weight", H, H, 3), b) if conv else att @ W(p + ".linear1.weight", H, H).t() + b
    x = x + mod[2] * o
    return x + mod[5] * _swiglu(W, p + ".ffn", _ln(x, mod[3], mod[4], s.ln_eps), H, s.F, conv)


def _exact_ref(case, inp):
    s, W = _spec(case), _Named(case)
    H, T, C, TS, out = s.H, s.T, s.C, s.TS, []
    for b in range(s.B):
        te = _sinusoid(inp["t"][b], H, s.t_max_period) @ W("t_embed.mlp.0.weight", H, H).t() + W("t_embed.mlp.0.bias")
        gc = _silu(te) @ W("t_embed.mlp.2.weight", H, H).t() + W("t_embed.mlp.2.bias") + inp["gcmlp"][b].to(F64)
        ext, gs = _silu(inp["sync"][b].to(F64) + gc), _silu(gc)
        x = _silu(_conv(inp["x"][b].to(F64), W("audio_input_proj.0.weight", H, s.latent, 3), W("audio_input_proj.0.bias")))
        xs = [_swiglu(W, "audio_input_proj.2", x, H, s.F, True), inp["clip"][b].to(F64), inp["text"][b].to(F64)]
        rope = [(1.0, T), (float(T) / C, C), None]
        for i in range(s.n_joint):
            last = i == s.n_joint - 1
            p = ["joint_blocks.%d.%s_block" % (i, n) for n in ("latent", "clip", "text")]
            mods = [_mod(W, p[j], ext if j == 0 else gs, 2 if last and j else 6, H) for j in range(3)]
            q, k, v = (torch.cat(t) for t in zip(*(_stream_qkv(W, p[j], s, xs[j], mods[j], rope[j], True) for j in range(3))))
            att = _attend(q, k, v, 0.125).split([T, C, TS])
            xs = [xs[j] if last and j else _ref_post(W, p[j], s, xs[j], att[j], mods[j], j < 2) for j in range(3)]
        x = xs[0]
        for i in range(s.n_fused):
            p = "fused_blocks.%d" % i
            mod = _mod(W, p, ext, 6, H)
            x = _ref_post(W, p, s, x, _attend(*_stream_qkv(W, p, s, x, mod, rope[0], True), 0.125), mod, True)
        m = _mod(W, "final_layer", ext, 2, H)
        out.append(_conv(_ln(x, m[0], m[1], s.ln_eps), W("final_layer.conv.weight", s.latent, H, 7), W("final_layer.conv.bias")))
    return {"flow": torch.stack(out)}


def _exact_cond(case, inp):
    s, W = _spec(case), _Named(case)
    H, F, SS = s.H, s.F, s.sync_S
    pos = W("sync_pos_emb", 8, s.sync_dim).repeat((SS + 7) // 8, 1)[:SS]
    x = _conv(inp["sync_f"].to(F64) + pos, W("sync_input_proj.0.weight", H, s.sync_dim, 7), W("sync_input_proj.0.bias"))
    x = _swiglu(W, "sync_input_proj.2", _silu(x), H, F, True)
    rows = np.floor((np.arange(s.T, dtype=np.float32) + np.float32(0.5)) * np.float32(SS) / np.float32(s.T)).astype(np.int64)
    out = {"sync_gather": x[torch.from_numpy(rows).to(DEV)]}
    c = _silu(inp["clip_f"].to(F64) @ W("clip_input_proj.0.weight", H, s.clip_dim).t() + W("clip_input_proj.0.bias"))
    out["clip_pp"] = _swiglu(W, "clip_input_proj.2", c, H, F, True)
    out["clip_fc"] = out["clip_pp"].mean(0) @ W("clip_cond_proj.weight", H, H).t() + W("clip_cond_proj.bias")
    for a in range(2):
        t = _silu(inp["text_cat"][a].to(F64) @ W("text_input_proj.0.weight", H, s.text_dim).t() + W("text_input_proj.0.bias"))
        out["text_pp%d" % a] = _swiglu(W, "text_input_proj.2", t, H, F, False)
        g = inp["gtext"][a].to(F64) @ W("text_cond_proj.weight", H, s.gtext_dim).t() + W("text_cond_proj.bias") + out["clip_fc"]
        out["gcmlp%d" % a] = _swiglu(W, "global_cond_mlp", g, H, F, False)
    return out


def _exact_clip(case, inp):
    s, W = _spec(case), _Named(case)
    n, H, ids = s.ctx, s.H, torch.from_numpy(inp["ids"].astype(np.int64)).to(DEV)
    off, _ = W.at["tok_emb"]
    x = W.flat[off:off + s.vocab * H].view(s.vocab, H)[ids].to(F64) + W("pos_emb", n, H)
    eot = int(np.argmax(inp["ids"]))
    r = torch.arange(n, device=DEV)
    keep = (r[None, :] <= r[:, None]) & (r[None, :] <= eot)
    bias = torch.where(keep, 0.0, -math.inf).to(F64)[None]

    def ln(x, p):
        c = x - x.mean(-1, keepdim=True)
        return c / (c.square().mean(-1, keepdim=True) + s.eps).sqrt() * W(p + ".w") + W(p + ".b")

    def lin(x, p, N, K):
        return x @ W(p + ".w", N, K).t() + W(p + ".b")

    for i in range(s.NL):
        b = "blk.%d" % i
        y = ln(x, b + ".ln1")
        q, k, v = (lin(y, b + t, H, H).reshape(n, s.NH, 64) for t in (".q", ".k", ".v"))
        x = x + lin(_attend(q, k, v, 0.125, bias), b + ".out", H, H)
        h = lin(ln(x, b + ".ln2"), b + ".fc1", 4 * H, H)
        x = x + lin(h * torch.sigmoid(1.702 * h), b + ".fc2", H, 4 * H)
    y = ln(x, "out_ln")
    return {"per_token": y, "pooled": y[eot] @ W("text_proj", H, H).t()}


def _exact_t5(case, inp):
    s, W = _spec(case), _Named(case)
    n, d, F, ids = s.ctx, s.d, s.d_ff, torch.from_numpy(inp["ids"].astype(np.int64)).to(DEV)
    off, _ = W.at["tok_emb"]
    x = W.flat[off:off + s.vocab * d].view(s.vocab, d)[ids].to(F64)
    # relative buckets: half of them per sign, exact up to half of that, logarithmic to max_dist
    half = s.n_bucket // 2
    exact = half // 2
    idx = np.empty((n, n), np.int64)
    for q in range(n):
        for k in range(n):
            a = abs(k - q)
            if a >= exact:
                a = min(half - 1, exact + int(math.log(a / exact) / math.log(s.max_dist / exact) * (half - exact)))
            idx[q, k] = a + (half if k > q else 0)
    bias = W("rel_bias", s.n_bucket, s.NH)[torch.from_numpy(idx).to(DEV)].permute(2, 0, 1)
    bias = bias + torch.where(ids != 0, 0.0, -math.inf).to(F64)[None, None]
    for i in range(s.NL):
        b = "blk.%d" % i
        y = _rms(x, W(b + ".attn_norm"), s.eps)
        q, k, v = ((y @ W(b + t, d, d).t()).reshape(n, s.NH, 64) for t in (".q", ".k", ".v"))
        x = x + _attend(q, k, v, 1.0, bias) @ W(b + ".o", d, d).t()
        y = _rms(x, W(b + ".ffn_norm"), s.eps)
        u = y @ W(b + ".wi_0", F, d).t()
        h = 0.5 * u * (1.0 + torch.tanh((0.7978845608 * (u + 0.044715 * u ** 3)).clamp(-10.0, 10.0)))
        x = x + (h * (y @ W(b + ".wi_1", F, d).t())) @ W(b + ".wo", d, F).t()
    return {"per_token": _rms(x, W("out_norm"), s.eps)}


def _exact_vae(case, inp):
    s, W = _spec(case), _Named(case)

    def snake(x, p):
        return x + (x * W(p + ".alpha").exp()).sin().square() * (-W(p + ".beta")).exp()

    x = _conv(inp["latent"].to(F64), W("decoder.layers.0.weight", s.width[0], s.latent, 7), W("decoder.layers.0.bias"))
    for n in range(5):
        p, st, K, ci, co = "decoder.layers.%d" % (n + 1), s.stride[n], s.kt[n], s.width[n], s.width[n + 1]
        h, w = snake(x, p + ".layers.0"), W(p + ".layers.1.weight", co, ci, K)
        T = h.shape[0]
        y = torch.zeros((T + 1) * st + 2 * K, co, device=DEV, dtype=F64)   # row r + K is output r
        pad = K - 1 - st // 2
        for k in range(K):   # input row u lands on output u * st + pad - k
            y[K + pad - k:K + pad - k + T * st:st] += h @ w[:, :, k].t()
        x = y[K:K + T * st] + W(p + ".layers.1.bias")
        for r in range(3):
            q = p + ".layers.%d" % (r + 2)
            g = _conv(snake(x, q + ".layers.0"), W(q + ".layers.1.weight", co, co, 7), W(q + ".layers.1.bias"), (1, 3, 9)[r])
            x = x + snake(g, q + ".layers.2") @ W(q + ".layers.3.weight", co, co).t() + W(q + ".layers.3.bias")
    return {"audio": _conv(snake(x, "decoder.layers.6"), W("decoder.layers.7.weight", s.out_ch, s.width[5], 7))}


def exact(case, seed):
    inp, k = _inputs(case, seed), case["kind"]
    if k == "tmlp":
        W0, b0, W2, b2, x, pooled = (inp[n].to(F64) for n in ("W0", "b0", "W2", "b2", "x", "pooled"))
        h = _silu(W0 @ x + b0)
        emb = W2 @ h + b2
        return {"h": h, "emb": emb, "g": _silu(pooled + emb)}
    if k == "gemm":
        y = inp["X"].to(F64) @ inp["W"].to(F64).t()
        return {"y": y if inp["b"] is None else y + inp["b"].to(F64)}
    if k == "attention":
        q, kk, v = inp["qkv"].to(F64).reshape(case["S"], 3, case["nh"], 64).unbind(1)
        return {"y": _attend(q, kk, v, 0.125)}
    return {"block": _exact_dit, "dit": _exact_dit, "ref": _exact_ref, "cond": _exact_cond, "clip": _exact_clip,
            "t5": _exact_t5, "vae": _exact_vae}[k](case, inp)
