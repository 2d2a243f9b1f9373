"""The work that programs using this library have it do, as cases that can be
timed and checked: the projections, the SSD scan, whole prefills and decode
steps, over the model shapes, weight formats and dtypes of lite_ssm_amd.model.

A case is a dict of plain values with a "kind":

  linear         lssm_linear: one projection of a prefill's rows (or of a larger
                 decode batch), residual added for out_proj
  decode_linear  lssm_norm_linear_decode: RMSNorm + projection of 1..64 rows, one
                 token of each sequence (in_proj, out_proj with its residual,
                 and the lm_head behind norm_f)
  ssd            lssm_ssd_chunked: the scan of a layer's prefill, state in and out
  prefill        Engine.reset + Engine.prefill: whole prompts to logits and states
  decode         Engine.decode_graph: greedy steps from a prefilled state

The single ops are enqueued inside a batch that stays open, as a forward pass
enqueues its layers' ops and commits once; the engine calls synchronise
themselves, as they do for every caller.  2.7B and 8B engines run a few of
their layers in front of the full vocabulary: through all 64 a rounding
difference in one layer grows past what 16-bit logits can be compared to.
"""
import ctypes
import functools
import math

import torch

import lite_ssm_amd as L
from lite_ssm_amd.model import DeviceModel, Engine, quantize, shape

ACT = {"f16": L.F16, "bf16": L.BF16, "f32": L.F32}
DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
FMT = {"dense": L.W_DENSE, "int4-b32": L.W_Q4_B32, "int4-g64": L.W_Q4_G64, "int8-g32": L.W_Q8_G32}
GROUP = {"int4-b32": 32, "int4-g64": 64, "int8-g32": 32}
MODELS = ("mamba2-130m", "mamba2-2.7b", "mamba2-8b")
LAYERS = {"mamba2-130m": 24, "mamba2-2.7b": 4, "mamba2-8b": 2}
EPS, DT_MIN, DT_MAX, CHUNK = 1e-5, 1e-6, 1e6, 64
# work limits of a drawn case: multiply-adds of a projection or prefill, bytes
# of a decode run
MAX_MACS, MAX_MACS_F32, MAX_BYTES = 4.4e11, 6e9, 1.2e10


def listed():
    return [
        # a one-paragraph prompt's rows through the 2.7B in_proj: too few for
        # full tiles, too many for the decode kernels
        dict(name="linear_prompt_100", kind="linear", model="mamba2-2.7b", layer="in_proj", rows=100,
             act="bf16", weights="int4-g64"),
        # unquantized half weights, the reference's own format, on a mid-size
        # ragged prompt of the widest model
        dict(name="linear_dense_777", kind="linear", model="mamba2-8b", layer="out_proj", rows=777,
             act="f16", weights="dense"),
        # fp32 model, as run to check a converted checkpoint against its source
        dict(name="linear_fp32_300", kind="linear", model="mamba2-130m", layer="in_proj", rows=300,
             act="f32", weights="dense"),
        # the smallest call: one token's out_proj of the smallest model
        dict(name="decode_linear_1", kind="decode_linear", model="mamba2-130m", layer="out_proj", rows=1,
             act="f16", weights="int8-g32"),
        # a serving batch that is not a power of two, int8 weights in bf16
        dict(name="decode_linear_24", kind="decode_linear", model="mamba2-8b", layer="in_proj", rows=24,
             act="bf16", weights="int8-g32"),
        # the vocabulary projection of a serving batch (never quantized)
        dict(name="lm_head_16", kind="decode_linear", model="mamba2-2.7b", layer="lm_head", rows=16,
             act="bf16", weights="dense"),
        # the fp32 scan of the 130M layer at 512 tokens
        dict(name="ssd_fp32_512", kind="ssd", model="mamba2-130m", batch=1, tokens=512, act="f32"),
        # the scan of a batch of long prompts
        dict(name="ssd_4x4096", kind="ssd", model="mamba2-2.7b", batch=4, tokens=4096, act="bf16"),
        # time to the first token of a short prompt, whole small model
        dict(name="prefill_130m_37", kind="prefill", model="mamba2-130m", layers=24, batch=1, tokens=37,
             act="f16", weights="int8-g32"),
        # a ragged prompt of some hundred tokens through layers of the 2.7B
        dict(name="prefill_2.7b_700", kind="prefill", model="mamba2-2.7b", layers=4, batch=1, tokens=700,
             act="bf16", weights="int4-g64"),
        # the largest: a batch of long prompts through the same layers
        dict(name="prefill_2.7b_4x4096", kind="prefill", model="mamba2-2.7b", layers=4, batch=4, tokens=4096,
             act="bf16", weights="int4-g64"),
        # a serving batch's decode through layers of the 2.7B
        dict(name="decode_2.7b_16", kind="decode", model="mamba2-2.7b", layers=4, batch=16, steps=4,
             act="bf16", weights="int4-g64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the same ranges.  Sizes over their logarithm; fp32 on the
    smallest model only (the others are not run in it)."""
    kind = rng.choice(("linear", "linear", "decode_linear", "decode_linear", "ssd", "prefill", "prefill", "decode"))
    act = rng.choice(("bf16", "bf16", "bf16", "f16", "f16", "f16", "f32"))
    model = "mamba2-130m" if act == "f32" else rng.choice(MODELS)
    weights = rng.choice(("dense", "int4-b32", "int4-g64", "int8-g32"))
    s = shape(model)
    if kind == "linear":
        layer = rng.choice(("in_proj", "out_proj"))
        macs = (s.proj if layer == "in_proj" else s.d_inner) * s.d_model
        most = min(16384, int((MAX_MACS_F32 if act == "f32" else MAX_MACS) / macs))
        return dict(kind=kind, model=model, layer=layer, rows=_log_int(rng, 5, most), act=act, weights=weights)
    if kind == "decode_linear":
        layer = rng.choice(("in_proj", "out_proj", "lm_head"))
        return dict(kind=kind, model=model, layer=layer, rows=_log_int(rng, 1, 64), act=act,
                    weights="dense" if layer == "lm_head" else weights)
    if kind == "ssd":
        batch = _log_int(rng, 1, 8)
        most = 2048 if act == "f32" else {"mamba2-130m": 16384, "mamba2-2.7b": 16384, "mamba2-8b": 8192}[model]
        return dict(kind=kind, model=model, batch=batch, tokens=_log_int(rng, 2, most // batch), act=act)
    if kind == "prefill":
        batch = _log_int(rng, 1, 4)
        macs = LAYERS[model] * s.linear_params()
        most = min(4096, int((MAX_MACS_F32 if act == "f32" else MAX_MACS) / macs))
        return dict(kind=kind, model=model, layers=LAYERS[model], batch=batch,
                    tokens=_log_int(rng, 1, max(2, most // batch)), act=act, weights=weights)
    case = dict(kind=kind, model=model, layers=LAYERS[model], batch=_log_int(rng, 1, 8 if act == "f32" else 64),
                steps=1, act=act, weights=weights)
    return dict(case, steps=min(_log_int(rng, 1, 16), max(1, int(MAX_BYTES / work(case)["bytes"]))))


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1 + seed)


def _randn(g, *size):
    return torch.randn(*size, generator=g, device="cuda")


def _linear_dims(case):
    s = shape(case["model"])
    return {"in_proj": (s.proj, s.d_model), "out_proj": (s.d_model, s.d_inner),
            "lm_head": (s.vocab_size, s.d_model)}[case["layer"]]


def _linear_inputs(case, seed):
    g, dt = _gen(seed), DTYPE[case["act"]]
    N, K = _linear_dims(case)
    M = case["rows"]
    w32 = (_randn(g, N, K) * 0.02).to(torch.float16).float()
    w, s = (w32.to(dt), None) if case["weights"] == "dense" else quantize(w32, FMT[case["weights"]])
    return dict(w=w, s=s, x=_randn(g, M, K).to(dt), norm_w=(1 + 0.1 * _randn(g, K)).to(dt),
                res=_randn(g, M, N).to(dt) if case["layer"] == "out_proj" else None)


def _ssd_inputs(case, seed):
    """X, B, C as the conv's SiLU leaves them in scale; dt, A and D as Mamba-2 sets them up."""
    g, dt = _gen(seed), DTYPE[case["act"]]
    s, b, n = shape(case["model"]), case["batch"], case["tokens"]
    H, P, G, N = s.n_heads, s.d_head, s.n_groups, s.d_state
    step = torch.exp(torch.rand(H, generator=g, device="cuda") * math.log(100.0) + math.log(1e-3))
    return dict(X=_randn(g, b, n, H, P).to(dt), B=(_randn(g, b, n, G, N) / N ** 0.5).to(dt),
                C=(_randn(g, b, n, G, N) / N ** 0.5).to(dt), dt=(0.5 * _randn(g, b, n, H)).to(dt),
                dt_bias=(step + torch.log(-torch.expm1(-step))).to(dt),
                A_log=torch.log(1 + 15 * torch.rand(H, generator=g, device="cuda")).to(dt),
                D=(1 + 0.1 * _randn(g, H)).to(dt), state=_randn(g, b, H, P, N))


def _model(case, seed):
    """A decode model's head predicts another token than its input with a wide
    margin, so that greedy ids do not hang on the last bits."""
    s = shape(case["model"], n_layer=case["layers"])
    how = dict(embed_std=1.0, head="permuted") if case["kind"] == "decode" else {}
    return DeviceModel(s, act=ACT[case["act"]], wfmt=FMT[case["weights"]], seed=seed, **how)


def _prompts(case, seed):
    g = torch.Generator().manual_seed(seed)
    n = case["tokens"] if case["kind"] == "prefill" else 32
    return torch.randint(0, shape(case["model"]).vocab_size, (case["batch"], n), generator=g,
                         dtype=torch.int32).cuda()


class _DeviceArray:
    """A buffer of `owner`, which lives as long as a tensor over the buffer does."""

    def __init__(self, owner, ptr, dims, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=dims, typestr=typestr, data=(ptr, False), version=2)


def _view(eng, ptr, dims, act):
    """A tensor over a buffer of the engine (no copy); it keeps the engine alive."""
    if act == "f32":
        return torch.as_tensor(_DeviceArray(eng, ptr, dims, "<f4"), device="cuda")
    return torch.as_tensor(_DeviceArray(eng, ptr, dims, "<i2"), device="cuda").view(DTYPE[act])


def _engine_outputs(eng, case):
    s, b, act = eng.model.shape, case["batch"], case["act"]
    p, c, h = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    L.check(L.lib.lssm_engine_logits(eng.h, ctypes.byref(p)))
    L.check(L.lib.lssm_engine_state(eng.h, ctypes.byref(c), ctypes.byref(h)))
    return dict(logits=_view(eng, p.value, (b, s.vocab_size), act),
                conv=_view(eng, c.value, (s.n_layer, b, s.xbc, s.d_conv), act),
                ssd=_view(eng, h.value, (s.n_layer, b, s.n_heads, s.d_head, s.d_state), "f32"))


@functools.lru_cache(None)
def _stream():
    """The program's one stream: passes follow each other, whatever state they are on."""
    return torch.cuda.Stream()


def prepare(case, seed):
    kind, act = case["kind"], ACT[case["act"]]
    ctx = L.Ctx(stream=_stream().cuda_stream)
    if kind in ("linear", "decode_linear"):
        N, K = _linear_dims(case)
        st = dict(_linear_inputs(case, seed), y=torch.empty(case["rows"], N, dtype=DTYPE[case["act"]], device="cuda"),
                  dims=(case["rows"], N, K), fmt=FMT[case["weights"]],
                  epi=L.EPI_ADD if case["layer"] == "out_proj" else L.EPI_NONE)
    elif kind == "ssd":
        s = shape(case["model"])
        st = dict(_ssd_inputs(case, seed), batch=case["batch"],
                  dims=L.SSDDims(case["tokens"], s.n_heads, s.d_head, s.d_state, s.n_groups,
                                 min(CHUNK, case["tokens"]), DT_MIN, DT_MAX, 1))
        st["Y"] = torch.empty_like(st["X"])
    else:
        model, ids = _model(case, seed), _prompts(case, seed)
        torch.cuda.synchronize()
        eng = Engine(ctx, model, case["batch"], ids.shape[1])
        st = dict(eng=eng, ids=ids, next=torch.zeros(case["batch"], dtype=torch.int32, device="cuda"),
                  out=_engine_outputs(eng, case), steps=case.get("steps"))
        torch.cuda.synchronize()
        if kind == "decode":
            eng.prefill(ids, st["next"])
    torch.cuda.synchronize()
    if "eng" not in st:
        ctx.begin_batch()
    return dict(st, kind=kind, ctx=ctx, act=act)


def run(st):
    kind, ctx = st["kind"], st["ctx"]
    if kind == "linear":
        ctx.linear(st["x"], st["w"], st["s"], st["y"], *st["dims"], st["fmt"], st["act"], st["epi"], st["res"])
        return st["y"]
    if kind == "decode_linear":
        s, r = st["s"], st["res"]
        L.check(L.lib.lssm_norm_linear_decode(
            ctx.h, st["x"].data_ptr(), st["norm_w"].data_ptr(), EPS, st["w"].data_ptr(),
            None if s is None else s.data_ptr(), st["y"].data_ptr(), None if r is None else r.data_ptr(),
            *st["dims"], st["fmt"], st["act"], st["epi"]))
        return st["y"]
    if kind == "ssd":
        ctx.ssd_chunked(st["X"], st["B"], st["C"], st["dt"], st["dt_bias"], st["A_log"], st["D"], st["Y"],
                        st["state"], st["batch"], st["dims"], st["act"])
        return dict(y=st["Y"], state=st["state"])
    eng = st["eng"]
    if kind == "prefill":
        eng.reset()
        eng.prefill(st["ids"], st["next"])
    else:
        eng.decode_graph(st["next"], st["next"], st["steps"])
    return st["out"]


# --------------------------------------------------------------------------- work, tolerance
def _weight_bytes(N, K, weights, act):
    if weights == "dense":
        return N * K * (4 if act == "f32" else 2)
    return N * K * (1.0 if weights == "int8-g32" else 0.5) + 2.0 * N * K / GROUP[weights]


def work(case):
    kind, act, s = case["kind"], case["act"], shape(case["model"])
    es = 4 if act == "f32" else 2
    state = s.n_heads * s.d_head * s.d_state           # of one layer and sequence
    if kind in ("linear", "decode_linear"):
        N, K = _linear_dims(case)
        M, res = case["rows"], case["layer"] == "out_proj"
        return dict(bytes=_weight_bytes(N, K, case["weights"], act) + es * M * (K + N * (2 if res else 1)),
                    flops=2.0 * M * N * K)
    if kind == "ssd":
        T = case["batch"] * case["tokens"]
        return dict(bytes=es * T * (2 * s.d_inner + 2 * s.n_groups * s.d_state + s.n_heads) + 8.0 * case["batch"] * state,
                    flops=4.0 * T * state)
    n, b = case["layers"], case["batch"]
    weights = n * (_weight_bytes(s.proj, s.d_model, case["weights"], act) +
                   _weight_bytes(s.d_model, s.d_inner, case["weights"], act)) + s.vocab_size * s.d_model * es
    per_token = n * (2.0 * s.linear_params() + 4.0 * state)
    head = 2.0 * s.vocab_size * s.d_model * b
    states = n * b * (4.0 * state + es * s.xbc * s.d_conv)
    if kind == "prefill":
        T = b * case["tokens"]
        return dict(bytes=weights + states + es * (T * s.d_model + b * s.vocab_size), flops=per_token * T + head)
    return dict(bytes=case["steps"] * (weights + 2 * states + es * b * s.vocab_size),
                flops=case["steps"] * (per_token * b + head))


def tolerance(case):
    """About four times the error against 64 bits seen per kind and type: one
    rounding of each output (and of the dequantized weights) in a projection;
    the state's rounding after every 64 tokens in a scan; every op's rounding
    in turn through an engine's layers."""
    if case["kind"] in ("linear", "decode_linear"):
        return {"rel": {"f16": 1.5e-3, "bf16": 1e-2, "f32": 2e-6}[case["act"]]}
    if case["kind"] == "ssd":
        return {"rel": {"f16": 3e-3, "bf16": 1e-2, "f32": 7e-6}[case["act"]]}
    return {"rel": {"f16": 2e-2, "bf16": 3e-2, "f32": 2e-5}[case["act"]]}


# --------------------------------------------------------------------------- the same in 64 bits
def _dense64(w, s, weights):
    if weights == "dense":
        return w.double()
    n = w.shape[0]
    if weights == "int8-g32":
        q = w.view(torch.int8).double()
    else:
        b = w.to(torch.int16)
        q = torch.stack([b & 15, b >> 4], -1).reshape(n, -1)
        q = torch.where(q >= 8, q - 16, q).double()
    g = GROUP[weights]
    return (q.reshape(n, -1, g) * s.double().reshape(n, -1, 1)).reshape(n, -1)


def _rms64(x, w):
    return x * w.double() / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)


def _ssd64(X, B, C, dt, dt_bias, A_log, D, S):
    """X [b, n, H, P], B / C [b, n, G, N], dt [b, n, H], S [b, H, P, N], all
    doubles: the recurrence s = e^{A dt} s + dt B x, y = C.s + D x, 64 tokens
    at a time."""
    n, H, G = X.shape[1], X.shape[2], B.shape[2]
    dt = torch.clamp(torch.nn.functional.softplus(dt + dt_bias, threshold=1e9), DT_MIN, DT_MAX)
    a = -torch.exp(A_log) * dt
    ys = []
    for t in range(0, n, CHUNK):
        x, d = X[:, t:t + CHUNK].transpose(1, 2), dt[:, t:t + CHUNK].transpose(1, 2)
        b, c = (v[:, t:t + CHUNK].transpose(1, 2).repeat_interleave(H // G, 1).contiguous() for v in (B, C))
        cum = a[:, t:t + CHUNK].transpose(1, 2).cumsum(-1)                       # [b, H, l]
        decay = torch.exp(torch.clamp(cum[..., :, None] - cum[..., None, :], max=0.0)).tril()
        m = torch.matmul(c, b.transpose(-1, -2).contiguous()) * decay * d[..., None, :]
        y = torch.matmul(m, x.contiguous()) + torch.exp(cum)[..., None] * torch.matmul(c, S.transpose(-1, -2).contiguous())
        ys.append(y.transpose(1, 2))
        w = torch.exp(cum[..., -1:] - cum) * d
        S = torch.exp(cum[..., -1])[..., None, None] * S + torch.matmul((x * w[..., None]).transpose(-1, -2).contiguous(), b)
    return torch.cat(ys, 1) + D[:, None] * X, S


def _layer64(s, w, weights, h, conv, S):
    """One mixer layer on h [b, n, d_model], continuing conv [b, xbc, K] and S."""
    b, n, K = h.shape[0], h.shape[1], s.d_conv
    proj = _rms64(h, w["norm_w"]) @ _dense64(w["in_proj_w"], w["in_proj_s"], weights).T
    z, xbc, dt = proj.split([s.d_inner, s.xbc, s.n_heads], -1)
    rows = torch.cat([conv.transpose(1, 2), xbc], 1)                              # K earlier rows, then the new
    cw = w["conv1d_w"].double()
    u = sum(rows[:, 1 + k:1 + k + n] * cw[:, k] for k in range(K)) + w["conv1d_b"].double()
    x, B, C = torch.nn.functional.silu(u).split([s.d_inner] + 2 * [s.n_groups * s.d_state], -1)
    y, S = _ssd64(x.reshape(b, n, s.n_heads, s.d_head), B.reshape(b, n, s.n_groups, s.d_state),
                  C.reshape(b, n, s.n_groups, s.d_state), dt, w["dt_bias"].double(), w["A_log"].double(),
                  w["D"].double(), S)
    g = _rms64(torch.nn.functional.silu(z) * y.reshape(b, n, s.d_inner), w["mixer_norm_w"])
    return h + g @ _dense64(w["out_proj_w"], w["out_proj_s"], weights).T, rows[:, -K:].transpose(1, 2), S


def _model64(case, seed):
    m, ids = _model(case, seed), _prompts(case, seed).long()
    s, b = m.shape, case["batch"]
    kw = dict(dtype=torch.float64, device="cuda")
    conv = [torch.zeros(b, s.xbc, s.d_conv, **kw) for _ in m.layers]
    ssd = [torch.zeros(b, s.n_heads, s.d_head, s.d_state, **kw) for _ in m.layers]

    def forward(tokens):
        h = m.embed[tokens].double()
        for i, w in enumerate(m.layers):
            h, conv[i], ssd[i] = _layer64(s, w, case["weights"], h, conv[i], ssd[i])
        return _rms64(h[:, -1], m.norm_f) @ m.lm_head.double().T

    logits = forward(ids)
    for _ in range(case.get("steps", 0)):
        logits = forward(logits.argmax(-1, keepdim=True))
    return dict(logits=logits, conv=torch.stack(conv), ssd=torch.stack(ssd))


def exact(case, seed):
    if case["kind"] in ("prefill", "decode"):
        return _model64(case, seed)
    if case["kind"] == "ssd":
        v = {k: t.double() for k, t in _ssd_inputs(case, seed).items()}
        y, S = _ssd64(v["X"], v["B"], v["C"], v["dt"], v["dt_bias"], v["A_log"], v["D"], v["state"])
        return dict(y=y, state=S)
    v = _linear_inputs(case, seed)
    x = v["x"].double()
    if case["kind"] == "decode_linear":
        x = _rms64(x, v["norm_w"])
    y = x @ _dense64(v["w"], v["s"], case["weights"]).T
    return y if v["res"] is None else y + v["res"].double()
