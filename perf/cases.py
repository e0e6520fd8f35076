"""Performance cases: the work that a user of this package has it do, through its public entry points.

A case is a dict of plain values.  Four kinds of work exist:

  decode   one `Session.forward` per step for `batch` sequences of one token each, as a serving loop calls it (the next
           tokens come from the host, the logits stay on the device), `steps` steps
  prefill  `batch` prompts of `tokens` tokens each through `Session.forward` in chunks of at most `chunk` tokens
  wkv      the WKV7 operator alone (`hip.wkv7`, or `hip.wkv7_f16state` for the fp16 state)
  sample   the device sampler alone (`hip.sample`) over `batch` rows of `vocab` logits, repetition penalties on

Model shapes are the package's presets at full depth with random-init weights; `fmt` is the weight format and `state`
the type of the WKV state.  `run` returns the logits (or the operator's output) and the whole updated state.

The functions: listed() -> cases; draw(rng) -> one more case of the same ranges; prepare(case, seed) -> what a program
holds before the call; run(state) -> outputs of one pass; work(case) -> bytes and operations a pass cannot do without;
tolerance(case) -> how far another correct implementation of the same precision may be off.
"""
import numpy as np
import torch

from rwkv_lightning_cuda_amd import hip
from rwkv_lightning_cuda_amd.model import PRESETS, HipModel, Session, State

FMTS = {"f16": hip.FMT_F16, "w8": hip.FMT_W8, "w4": hip.FMT_W4}
# standard deviation of the WKV state after a few hundred tokens of these random-init models
STATE_STD = {"0.1B": 0.25, "1.5B": 0.9, "7.2B": 2.0}


def listed():
    return [
        # the operator of the smallest model on a short text, fp32 tensors: a handful of microseconds, all latency
        dict(name="wkv op, one short text", kind="wkv", batch=1, tokens=64, heads=12, io="f32", state="f32"),
        # the operator on a batch of long documents
        dict(name="wkv op, long batch", kind="wkv", batch=16, tokens=2048, heads=64, io="f16", state="f32"),
        # the sampler of a full serving batch with every filter on
        dict(name="sampler, 64 rows", kind="sample", batch=64, vocab=65536, top_k=50, top_p=0.6),
        # one user on the smallest model: launches and latency
        dict(name="decode 0.1B f16 b1", kind="decode", preset="0.1B", fmt="f16", state="f32", batch=1, steps=4),
        # a small server: the middle model, an odd number of live sequences, the server's default state type
        dict(name="decode 1.5B w8 b13", kind="decode", preset="1.5B", fmt="w8", state="f16", batch=13, steps=4),
        # one user on the large model, the two quantised formats
        dict(name="decode 7.2B w8 b1", kind="decode", preset="7.2B", fmt="w8", state="f32", batch=1, steps=4),
        dict(name="decode 7.2B w4 b2", kind="decode", preset="7.2B", fmt="w4", state="f32", batch=2, steps=4),
        # a few users, and a full serving batch
        dict(name="decode 7.2B w8 b8", kind="decode", preset="7.2B", fmt="w8", state="f32", batch=8, steps=4),
        dict(name="decode 7.2B w8 b64", kind="decode", preset="7.2B", fmt="w8", state="f16", batch=64, steps=4),
        # one prompt in the default chunks (the last one ragged)
        dict(name="prefill 7.2B w8 500", kind="prefill", preset="7.2B", fmt="w8", state="f32", batch=1, tokens=500, chunk=128),
        # a few prompts of odd length with unquantised weights, whole
        dict(name="prefill 1.5B f16 3x333", kind="prefill", preset="1.5B", fmt="f16", state="f32", batch=3, tokens=333,
             chunk=512),
        # a batch of prompts: the largest call
        dict(name="prefill 7.2B w8 16x128", kind="prefill", preset="7.2B", fmt="w8", state="f32", batch=16, tokens=128,
             chunk=128),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 4 + ["wkv", "sample"])
    if kind == "wkv":
        state = rng.choice(["f32", "f32", "f16"])
        io = "f16" if state == "f16" else rng.choice(["f16", "f16", "f32"])
        heads = rng.choice([12, 32, 64])
        batch = _log_int(rng, 1, 16)
        return dict(kind="wkv", batch=batch, tokens=_log_int(rng, 2, 2048), heads=heads, io=io, state=state)
    if kind == "sample":
        top_k, top_p = rng.choice([(0, 1.0), (50, 0.6), (0, 0.9), (rng.randint(2, 200), 1.0), (rng.randint(2, 200), 0.8)])
        return dict(kind="sample", batch=_log_int(rng, 1, 128), vocab=65536, top_k=top_k, top_p=top_p)
    preset = rng.choice(["0.1B", "1.5B", "7.2B", "7.2B"])
    fmt = "f16" if preset == "0.1B" else rng.choice(["w8", "w8", "w4", "f16"])
    state = rng.choice(["f32", "f16"])
    if kind == "decode":
        return dict(kind="decode", preset=preset, fmt=fmt, state=state, batch=_log_int(rng, 1, 128),
                    steps=rng.choice([2, 3, 5, 6]))
    rows = _log_int(rng, 8, 2048)
    batch = min(_log_int(rng, 1, 32), rows // 4)
    chunk = rng.choice([128, 512])
    return dict(kind="prefill", preset=preset, fmt=fmt, state=state, batch=batch, tokens=rows // batch, chunk=chunk)


# ---- inputs ---------------------------------------------------------------------------------------------------------
class _Memory:
    """torch's view of a device array of the package (no copy); the tensor keeps this object, and so the array, alive."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": array.dtype.str, "data": (array.ptr, False),
                                         "version": 3}


def _view(array):
    return torch.as_tensor(_Memory(array), device="cuda")


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


class _Program:
    """A model with its session, generation state and logits buffer; gives the device memory back when it goes."""

    def __init__(self, case, seed):
        dims = PRESETS[case["preset"]]
        B = case["batch"]
        self.kind = case["kind"]
        self.model = HipModel.random_on_device(dims, FMTS[case["fmt"]], seed=seed % 1000003)
        self.session = Session(self.model)
        self.state = State(dims, B, wkv_fp16=case["state"] == "f16")
        self.logits = hip.DeviceArray.zeros((B, dims.V), np.float32)
        self.outputs = {"logits": _view(self.logits), "shift": _view(self.state.shift), "wkv": _view(self.state.wkv),
                        "elapsed": _view(self.state.elapsed)}
        # every sequence has been read for a while already
        g = _generator(seed)
        out = self.outputs
        out["wkv"].normal_(0.0, STATE_STD[case["preset"]], generator=g)
        out["shift"].normal_(0.0, 1.0, generator=g)
        rng = np.random.default_rng(seed)
        out["elapsed"].copy_(torch.from_numpy(rng.integers(100, 3000, (B,)).astype(np.int32)))
        if self.kind == "decode":
            self.calls = list(rng.integers(0, dims.V, (case["steps"], B, 1)))
        else:
            tokens = rng.integers(0, dims.V, (B, case["tokens"]))
            self.calls = [tokens[:, i:i + case["chunk"]] for i in range(0, case["tokens"], case["chunk"])]
        torch.cuda.synchronize()

    def __del__(self):
        if hasattr(self, "session"):
            self.session.close()
        if hasattr(self, "model"):
            self.model.close()


def _prepare_wkv(case, seed):
    """r, k, v ~ N(0,1); decay = exp(-exp(U(-6,-0.5))) as its raw logit; a = -k/|k| per head, b = k/|k| * sigmoid(U(-3,3))."""
    B, T, H = case["batch"], case["tokens"], case["heads"]
    C = H * 64
    g = _generator(seed)
    io = torch.float16 if case["io"] == "f16" else torch.float32

    def normal():
        return torch.randn(B, T, C, generator=g, device="cuda")

    def uniform(lo, hi):
        return torch.rand(B, T, C, generator=g, device="cuda") * (hi - lo) + lo

    k = normal()
    kk = (k.view(B, T, H, 64) / k.view(B, T, H, 64).norm(dim=-1, keepdim=True)).view(B, T, C)
    s = torch.exp(uniform(-6.0, -0.5) + 0.5)
    t = {"r": normal(), "w": torch.log(s / (1.0 - s)), "k": k, "v": normal(), "a": -kk, "b": kk * torch.sigmoid(uniform(-3.0, 3.0))}
    t = {name: x.to(io).contiguous() for name, x in t.items()}
    t["y"] = torch.zeros(B, T, C, dtype=io, device="cuda")
    t["state"] = torch.zeros(B, H, 64, 64, dtype=torch.float16 if case["state"] == "f16" else torch.float32, device="cuda")
    t["elapsed"] = torch.randint(0, 3000, (B,), generator=g, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()
    return {"kind": "wkv", "case": dict(case), "t": t, "p": {name: x.data_ptr() for name, x in t.items()}}


def _prepare_sample(case, seed):
    B, V = case["batch"], case["vocab"]
    g = _generator(seed)
    t = {"logits": torch.randn(B, V, generator=g, device="cuda") * 3.0, "penalties": torch.zeros(B, V, device="cuda"),
         "probs": torch.zeros(B, V, device="cuda"), "picked": torch.zeros(B, dtype=torch.int32, device="cuda")}
    # the last tokens of every row carry a penalty already
    seen = torch.randint(0, V, (B, 64), generator=g, device="cuda")
    t["penalties"].scatter_(1, seen, torch.rand(B, 64, generator=g, device="cuda") + 0.5)
    torch.cuda.synchronize()
    return {"kind": "sample", "case": dict(case), "t": t, "p": {name: x.data_ptr() for name, x in t.items()}, "seed": seed}


def prepare(case, seed):
    if case["kind"] == "wkv":
        return _prepare_wkv(case, seed)
    if case["kind"] == "sample":
        return _prepare_sample(case, seed)
    return {"kind": case["kind"], "program": _Program(case, seed)}


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(state):
    if state["kind"] == "wkv":
        c, p = state["case"], state["p"]
        B, T, H = c["batch"], c["tokens"], c["heads"]
        if c["state"] == "f16":
            hip.wkv7_f16state(B, T, H * 64, H, p["state"], p["r"], p["w"], p["k"], p["v"], p["a"], p["b"], p["y"], p["elapsed"])
        else:
            hip.wkv7(B, T, H * 64, H, hip.W_RAW_LOGIT, hip.IO_F16 if c["io"] == "f16" else hip.IO_F32, p["state"], p["r"],
                     p["w"], p["k"], p["v"], p["a"], p["b"], p["y"])
        return {"y": state["t"]["y"], "state": state["t"]["state"]}
    if state["kind"] == "sample":
        c, p = state["case"], state["p"]
        hip.sample(c["batch"], c["vocab"], p["logits"], p["penalties"], p["probs"], p["picked"], presence=0.5, frequency=0.1,
                   decay=0.99, temperature=1.0, top_k=c["top_k"], top_p=c["top_p"], seed=state["seed"], step=0)
        return {"picked": state["t"]["picked"], "penalties": state["t"]["penalties"]}
    prog = state["program"]
    for tokens in prog.calls:
        prog.session.forward(tokens, prog.state, prog.logits)
    return prog.outputs


# ---- what a pass cannot do without, and how far results may be apart --------------------------------------------------
def work(case):
    if case["kind"] == "wkv":
        B, T, H = case["batch"], case["tokens"], case["heads"]
        n = B * T * H * 64
        return {"bytes": 7 * n * (2 if case["io"] == "f16" else 4) + 2 * B * H * 4096 * (2 if case["state"] == "f16" else 4),
                "flops": 10.0 * n * 64}
    if case["kind"] == "sample":
        # logits and penalties in, penalties out
        return {"bytes": 12 * case["batch"] * case["vocab"], "flops": 10.0 * case["batch"] * case["vocab"]}
    d = PRESETS[case["preset"]]
    B = case["batch"]
    dense = d.L * (4 * d.C * d.C + 2 * d.F * d.C)
    lora = 2 * d.C * (d.L * (d.Rw + d.Ra + d.Rg) + (d.L - 1) * d.Rv)
    head = d.V * d.C
    per = {"f16": 2.0, "w8": 1.0, "w4": 0.5 + 3.0 / 128}[case["fmt"]]
    weights = (dense + head) * per + lora * 2 + d.L * 19 * d.C * 2
    state = 2 * d.L * B * (d.H * 4096 * (2 if case["state"] == "f16" else 4) + 2 * d.C * 2)
    if case["kind"] == "decode":
        calls, tokens = case["steps"], case["steps"] * B
    else:
        calls, tokens = -(-case["tokens"] // case["chunk"]), B * case["tokens"]
    return {"bytes": calls * (weights + state + B * d.V * 4) + tokens * d.C * 2,
            "flops": 2.0 * (dense + lora) * tokens + 2.0 * head * B * calls + d.L * d.H * 4096 * 10.0 * tokens}


def tolerance(case):
    if case["kind"] == "wkv":
        # against 64-bit sums: 1.4e-3 with the fp16 state, 2.1e-4 (the rounding of y) with fp16 tensors, 1.1e-7 in fp32
        return {"rel": 6e-3} if case["state"] == "f16" else {"rel": 8e-4 if case["io"] == "f16" else 1e-6}
    if case["kind"] == "sample":
        return {"rel": 1e-6, "differ": 0.01}
    # the same calls with their sums in another order (other chunks, other kernels of the package): up to 5e-3 (6e-3 with
    # the fp16 state) of the state and 4e-3 of the logits, single values up to 0.09 of the root mean square
    return {"rel": 0.02, "max": 0.4}
