"""What a program that uses this library spends its GPU time on, as cases
that can be timed and compared.

A serving engine calls, per layer and step, one mixer (Gated DeltaNet or
gated GQA) between two projections: decode or verify steps over a batch of
sequences, prompt prefills, and the bf16 projections beside them. Each case
is one such call through the Python binding of the C ABI on device tensors.
Shapes are the model's (hidden 2048; GDN 16 K heads, 32 V heads of 128; GQA
16 query heads, 2 kv heads of 256), inputs are drawn with the distributions
of the repository's benchmark, and batch sizes, contexts and prompt lengths
cover what the library takes, ragged ones among them.
"""
import math
import os
import random
import sys

import numpy as np
import torch

PKG = os.path.join(os.getcwd(), "apus-qwen3.6-35b-a3b_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import apus_hip  # noqa: E402

HID = 2048
GDN = (16, 32, 128, 128)                   # K heads, V heads, dk, dv
HK, HV, DK, DV = GDN
KD, VD = HK * DK, HV * DV
CD = 2 * KD + VD                           # conv channels (q | k | v)
ATTN = (16, 2, 256, 64, 1e7)               # heads, kv heads, d, rotary dims, theta
NH, NKV, D, ROT, THETA = ATTN
GRP = NH // NKV
BLK = 32                                   # positions per KV block
EPS = 1e-6
BF = torch.bfloat16

# (outputs, inputs) of the model's projections: the GDN layer's fused input
# projection and its output projection, the attention layer's query|gate
# and key/value projections
PROJ = ((CD + VD + 2 * HV, HID), (HID, VD), (NH * 2 * D, HID), (NKV * D, HID))


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one user's chat step: a single token through a GDN layer, where
        # only latency counts
        dict(name="gdn_decode_1", kind="gdn_decode", seqs=1, most=1, slots=False, shape=0),
        # a serving batch verifying 1..4 speculative tokens per sequence,
        # states in a slot pool in shuffled order
        dict(name="gdn_verify_128", kind="gdn_decode", seqs=128, most=4, slots=True, shape=15),
        # a handful of prompts of chat length prefilled as one ragged batch
        dict(name="gdn_prefill_ragged", kind="gdn_prefill", seqs=6, tokens=997, shape=3),
        # one long prompt
        dict(name="gdn_prefill_4096", kind="gdn_prefill", seqs=1, tokens=4096, shape=0),
        # one user's chat step through a full-attention layer
        dict(name="attn_decode_1", kind="attn_decode", seqs=1, ctx=1500, most=1, spread=False,
             paged=False, shape=0),
        # the serving batch's verify step on a paged cache, contexts
        # log-normal around 4096
        dict(name="attn_verify_128", kind="attn_decode", seqs=128, ctx=4096, most=4, spread=True,
             paged=True, shape=15),
        # long-context decode: every sequence at 32K positions
        dict(name="attn_decode_64x32768", kind="attn_decode", seqs=64, ctx=32767, most=1,
             spread=False, paged=False, shape=0),
        # prompts continuing after cached prefixes of several lengths
        dict(name="attn_prefill_ragged", kind="attn_prefill", seqs=5, tokens=701, ctx=3000,
             paged=True, shape=4),
        # one long prompt from position 0
        dict(name="attn_prefill_8192", kind="attn_prefill", seqs=1, tokens=8192, ctx=0,
             paged=False, shape=0),
        # the bitwise projection of one token (the GDN input projection)
        dict(name="proj_exact_1", kind="proj", rows=1, outs=CD + VD + 2 * HV, ins=HID, exact=True),
        # the same projection of a long prompt
        dict(name="proj_4096", kind="proj", rows=4096, outs=CD + VD + 2 * HV, ins=HID,
             exact=False),
        # a GDN layer with its projections on the serving batch
        dict(name="gdn_layer_128", kind="layer", mixer="gdn", seqs=128, ctx=0, most=4, shape=15),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("gdn_decode", "gdn_prefill", "attn_decode", "attn_prefill", "proj",
                       "layer"))
    shape = rng.randrange(1, 1 << 16)
    if kind == "gdn_decode":
        return dict(kind=kind, seqs=_logu(rng, 1, 256), most=rng.randint(1, 4),
                    slots=rng.random() < 0.5, shape=shape)
    if kind == "gdn_prefill":
        seqs = _logu(rng, 1, 16)
        return dict(kind=kind, seqs=seqs, tokens=_logu(rng, 8, 8192 // seqs), shape=shape)
    if kind == "attn_decode":
        seqs = _logu(rng, 1, 128)
        spread = rng.random() < 0.5
        most_ctx = min(32768, (1 << 20) // seqs if spread else (2 << 20) // seqs)
        return dict(kind=kind, seqs=seqs, ctx=_logu(rng, 64, most_ctx), most=rng.randint(1, 4),
                    spread=spread, paged=rng.random() < 0.5, shape=shape)
    if kind == "attn_prefill":
        seqs = _logu(rng, 1, 8)
        tokens = _logu(rng, 8, int(8192 / math.sqrt(seqs)))
        room = max(1, (8192 * 8192 // (2 * seqs * tokens)) - tokens)
        ctx = 0 if rng.random() < 0.5 else _logu(rng, 16, max(16, min(8192, room)))
        return dict(kind=kind, seqs=seqs, tokens=tokens, ctx=ctx, paged=rng.random() < 0.5,
                    shape=shape)
    if kind == "proj":
        outs, ins = rng.choice(PROJ)
        if rng.random() < 0.25:
            return dict(kind=kind, rows=rng.randint(1, 8), outs=outs, ins=ins, exact=True)
        return dict(kind=kind, rows=_logu(rng, 1, 4096), outs=outs, ins=ins, exact=False)
    mixer = rng.choice(("gdn", "gdn", "gdn", "attn"))
    return dict(kind=kind, mixer=mixer, seqs=_logu(rng, 1, 128),
                ctx=_logu(rng, 64, 8192) if mixer == "attn" else 0, most=rng.randint(1, 4),
                shape=shape)


def _new_tokens(case):
    """New tokens of each sequence."""
    r, n = random.Random(case["shape"]), case["seqs"]
    if "tokens" in case:                   # prompts: the longest, then log-uniform ones
        return [case["tokens"]] + [_logu(r, 1, case["tokens"]) for _ in range(n - 1)]
    return [r.randint(1, case["most"]) for _ in range(n)]


def _cached(case):
    """Positions cached before the call, of each sequence."""
    r, n, ctx = random.Random(case["shape"] + 1), case["seqs"], case["ctx"]
    if case["kind"] == "attn_prefill":
        return [_logu(r, 1, ctx) if ctx else 0 for _ in range(n)]
    if case.get("spread", True) and n > 1:
        return [min(65000, max(16, ctx // 16, int(ctx * math.exp(r.gauss(0.0, 1.0)))))
                for _ in range(n)]
    return [ctx] * n


def _mixer(case):
    return case["mixer"] if case["kind"] == "layer" else case["kind"].split("_")[0]


# ----------------------------------------------------------------- inputs
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def bf(self, *shape, std=1.0, mean=0.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=BF)
        if std != 1.0:
            x.mul_(std)
        return x.add_(mean) if mean else x

    def f32(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda").mul_(std)

    def uniform(self, n, hi):
        return torch.rand(n, generator=self.g, device="cuda") * hi


_ready = False


def _init():
    global _ready
    if not _ready:
        apus_hip.init(0)
        apus_hip.set_stream(torch.cuda.current_stream().cuda_stream)
        _ready = True


def _gdn_inputs(case, R, s):
    n = s["new"] = _new_tokens(case)
    T, B = sum(n), len(n)
    s["cu"] = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    s["w"] = dict(conv_w=R.bf(CD, 4, std=0.1), A_log=R.uniform(HV, 2.7),
                  dt_bias=torch.ones(HV, device="cuda"), onorm_w=R.bf(DV, std=0.1, mean=1.0))
    s["layer"] = apus_hip.gdn_layer(GDN, s["w"])
    pooled = bool(case.get("slots")) or case["kind"] == "layer"
    nslot = B + 8 if pooled else B
    if case["kind"] == "gdn_prefill":      # a new prompt starts from zero state
        s["conv"] = torch.zeros((nslot, CD * 3), dtype=BF, device="cuda")
        s["S"] = torch.zeros((nslot, HV, DK * DV), device="cuda")
    else:
        s["conv"] = R.bf(nslot, CD * 3)
        s["S"] = R.f32(nslot, HV, DK * DV, std=0.02)
    order = list(range(nslot))
    if pooled:
        random.Random(case["shape"] + 2).shuffle(order)
    s["slot"] = np.array(order[:B], np.int32)
    s["pooled"] = pooled
    if case["kind"] == "layer":
        k = HID ** -0.5
        s["pw"] = dict(w_qkv=R.bf(CD, HID, std=k), w_z=R.bf(VD, HID, std=k),
                       w_b=R.bf(HV, HID, std=k), w_a=R.bf(HV, HID, std=k),
                       w_out=R.bf(HID, VD, std=VD ** -0.5))
        s["proj"] = apus_hip.gdn_proj(HID, s["pw"])
        s["ln1"] = R.bf(T, HID)
        s["out"] = torch.empty((T, HID), dtype=BF, device="cuda")
    else:
        s.update(qkv=R.bf(T, CD), z=R.bf(T, VD), a=R.bf(T, HV), b=R.bf(T, HV),
                 out=torch.empty((T, VD), dtype=BF, device="cuda"))
    if case["kind"] == "gdn_decode" and not pooled:
        # a decode loop on fixed buffers keeps the prepared call
        s["call"] = apus_hip.gdn_decode_bound(s["layer"], s["cu"], s["qkv"], s["z"], s["a"],
                                              s["b"], s["conv"], s["S"], s["out"])


def _attn_inputs(case, R, s):
    n = s["new"] = _new_tokens(case)
    ctx = s["ctx"] = _cached(case)
    T, B = sum(n), len(n)
    s["cu"] = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    s["pos0"] = np.array(ctx, np.int32)
    s["w"] = dict(qn_w=R.bf(D, std=0.1), kn_w=R.bf(D, std=0.1))
    s["layer"] = apus_hip.attn_layer(ATTN, s["w"])
    nblk = [-(-(c + k) // BLK) for c, k in zip(ctx, n)]
    s["paged"] = bool(case.get("paged")) or case["kind"] == "layer"
    width = max(nblk)
    s["max_seq"] = width * BLK
    if s["paged"]:                         # blocks handed out in any order
        ids = list(range(sum(nblk)))
        random.Random(case["shape"] + 3).shuffle(ids)
        table = np.zeros((B, width), np.int32)
        for i, k in enumerate(nblk):
            table[i, :k] = ids[:k]
            del ids[:k]
    else:
        table = np.arange(B * width, dtype=np.int32).reshape(B, width)
    total = sum(nblk) if s["paged"] else B * width
    s["table"], s["nblk"] = table, np.array(nblk, np.int32)
    s["k_cache"] = R.bf(total, NKV, BLK, D)
    s["v_cache"] = R.bf(total, NKV, D, BLK)
    if s["paged"]:
        s["table_dev"] = torch.from_numpy(table).to("cuda")
        s["rows"] = np.arange(B, dtype=np.int32)
        s["kv"] = apus_hip.KvCache(s["k_cache"].data_ptr(), s["v_cache"].data_ptr(),
                                   s["table_dev"].data_ptr(), width, B, s["nblk"].ctypes.data)
    if case["kind"] == "layer":
        k = HID ** -0.5
        s["pw"] = dict(wq=R.bf(NH * 2 * D, HID, std=k), wk=R.bf(NKV * D, HID, std=k),
                       wv=R.bf(NKV * D, HID, std=k), wo=R.bf(HID, NH * D, std=(NH * D) ** -0.5))
        s["proj"] = apus_hip.attn_proj(HID, s["pw"])
        s["ln1"] = R.bf(T, HID)
        s["out"] = torch.empty((T, HID), dtype=BF, device="cuda")
    else:
        s.update(qg=R.bf(T, NH, 2 * D), k=R.bf(T, NKV, D), v=R.bf(T, NKV, D),
                 out=torch.empty((T, NH * D), dtype=BF, device="cuda"))


def prepare(case, seed):
    _init()
    R = _Rand(seed)
    s = dict(case=case)
    if case["kind"] == "proj":
        s.update(wt=R.bf(case["outs"], case["ins"], std=case["ins"] ** -0.5),
                 x=R.bf(case["rows"], case["ins"]),
                 out=torch.empty((case["rows"], case["outs"]), dtype=BF, device="cuda"))
    elif _mixer(case) == "gdn":
        _gdn_inputs(case, R, s)
    else:
        _attn_inputs(case, R, s)
    return s


# -------------------------------------------------------------------- run
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "proj":
        apus_hip.bf16_gemm_dev(s["wt"], s["x"], s["out"], exact=case["exact"])
        return {"y": s["out"]}
    if _mixer(case) == "gdn":
        if kind == "layer":
            apus_hip.gdn_layer_decode_slots(s["layer"], s["proj"], s["slot"], s["slot"], s["cu"],
                                            s["ln1"], s["conv"].data_ptr(), s["S"].data_ptr(),
                                            s["out"])
        elif kind == "gdn_prefill":
            apus_hip.gdn_prefill(s["layer"], s["cu"], s["qkv"], s["z"], s["a"], s["b"], s["conv"],
                                 s["S"], s["out"])
        elif s["pooled"]:
            apus_hip.gdn_decode_slots(s["layer"], s["slot"], s["slot"], s["cu"], s["qkv"], s["z"],
                                      s["a"], s["b"], s["conv"].data_ptr(), s["S"].data_ptr(),
                                      s["out"])
        else:
            s["call"]()
        return {"y": s["out"], "conv": s["conv"], "S": s["S"]}
    if kind == "layer":
        apus_hip.attn_layer_decode_paged(s["layer"], s["proj"], s["rows"], s["cu"], s["pos0"],
                                         s["ln1"], s["kv"], s["out"])
    elif s["paged"]:
        f = apus_hip.attn_prefill_paged if kind == "attn_prefill" else apus_hip.attn_decode_paged
        f(s["layer"], s["rows"], s["cu"], s["pos0"], s["qg"], s["k"], s["v"], s["kv"], s["out"])
    else:
        f = apus_hip.attn_prefill if kind == "attn_prefill" else apus_hip.attn_decode
        f(s["layer"], s["cu"], s["pos0"], s["qg"], s["k"], s["v"], s["k_cache"], s["v_cache"],
          s["max_seq"], s["out"])
    return {"y": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


# ------------------------------------------------------------------- work
def work(case):
    if case["kind"] == "proj":
        M, O, K = case["rows"], case["outs"], case["ins"]
        return {"bytes": 2 * (M * K + O * K + M * O), "flops": 2 * M * O * K}
    n = _new_tokens(case)
    T, B = sum(n), len(n)
    layer = case["kind"] == "layer"
    if _mixer(case) == "gdn":
        state = HV * DK * DV * 4 * 2 + CD * 3 * 2 * 2      # read and written
        fixed = CD * 4 * 2 + HV * 4 * 2 + DV * 2           # conv, gate and norm weights
        per = CD * 2 + VD * 2 + HV * 2 * 2 + VD * 2        # qkv, z, a, b in, y out
        flops = T * HV * (7 * DK * DV)                     # decay, k S, update, q S
        if layer:
            fixed += ((CD + VD + 2 * HV) * HID + HID * VD) * 2
            per = 2 * HID * 2                              # ln1 in, ao out
            flops += 2 * T * HID * (CD + VD + 2 * HV + VD)
        return {"bytes": B * state + fixed + T * per, "flops": flops}
    ctx = _cached(case)
    keys = sum(c + k for c, k in zip(ctx, n))
    pairs = sum(k * c + k * (k + 1) // 2 for c, k in zip(ctx, n))
    # cached K and V read; the new positions' rows appended
    per = NH * 2 * D * 2 + 2 * NKV * D * 2 + 2 * NKV * D * 2 + NH * D * 2
    fixed = 2 * D * 2 + (keys - T) * NKV * D * 2 * 2
    flops = NH * 4 * D * pairs
    if layer:
        fixed += ((NH * 2 * D + 2 * NKV * D) * HID + HID * NH * D) * 2
        per = 2 * HID * 2 + 2 * NKV * D * 2
        flops += 2 * T * HID * (NH * 2 * D + 2 * NKV * D + NH * D)
    return {"bytes": fixed + T * per, "flops": flops}


def tolerance(case):
    """About four times the distance of each path from exact() below, which
    leaves the last rounding to bf16 out (2e-3 of a bf16 result). The
    reference-order projection is defined bit for bit."""
    if case["kind"] == "proj":
        return "exact" if case["exact"] else {"rel": 7e-3, "max": 0.05}
    return {"rel": 8e-3, "max": 0.15}


# ------------------------------------------------------------------ exact
# The same call in float64. Values that the operation defines as bf16
# tensors between its steps (conv output, attention scores and
# probabilities, the steps of the gated norm, a layer's projections) are
# rounded there; sums, products and functions are float64, and the result
# itself is left unrounded.
def _rnd(x):
    return x.to(BF).double()


def _sig(x):
    return 1.0 / (1.0 + torch.exp(-x))


def _unpack(S):
    """Device state layout -> [.., i, j]."""
    return S.reshape(-1, 2, 32, 64, 4).permute(0, 2, 4, 1, 3).reshape(-1, DK, DV)


def _pack(S):
    return S.reshape(-1, 32, 4, 2, 64).permute(0, 3, 1, 4, 2).reshape(-1, DK * DV)


def _exact_gdn(s, qkv, z, a, b):
    """(y, conv, S) of the GDN mixer for float64 inputs [T, ..]."""
    w, n, cu = s["w"], s["new"], s["cu"]
    B, longest = len(n), max(n)
    slot = torch.from_numpy(s["slot"].astype(np.int64)).to("cuda")
    conv, S = s["conv"].double(), s["S"].double()
    old = conv[slot].reshape(B, CD, 3)
    taps = w["conv_w"].double()
    pad = dict(device="cuda", dtype=torch.float64)
    q = torch.zeros(B, longest, HK, DK, **pad)
    k = torch.zeros(B, longest, HK, DK, **pad)
    v = torch.zeros(B, longest, HV, DV, **pad)
    dec = torch.ones(B, longest, HV, **pad)
    beta = torch.zeros(B, longest, HV, **pad)
    for i in range(B):
        r = slice(int(cu[i]), int(cu[i + 1]))
        x = torch.cat([old[i].t(), qkv[r]])                # [3 + n, CD]
        co = _rnd(sum(x[j:j + n[i]] * taps[:, j] for j in range(4)))
        c = _rnd(co * _sig(co))
        conv[slot[i]] = x[-3:].t().reshape(-1)

        def unit(h):
            return h / torch.sqrt(h.square().sum(-1, keepdim=True) + EPS)
        q[i, :n[i]] = unit(c[:, :KD].reshape(-1, HK, DK)) * DK ** -0.5
        k[i, :n[i]] = unit(c[:, KD:2 * KD].reshape(-1, HK, DK))
        v[i, :n[i]] = c[:, 2 * KD:].reshape(-1, HV, DV)
        t = a[r] + w["dt_bias"].double()
        dec[i, :n[i]] = torch.exp(-torch.exp(w["A_log"].double()) * torch.log1p(torch.exp(t)))
        beta[i, :n[i]] = _rnd(_sig(b[r]))
    St = _unpack(S[slot]).reshape(B, HV, DK, DV)
    o = torch.zeros(B, longest, HV, DV, **pad)
    rep = HV // HK
    for t in range(longest):                               # padding leaves S as it is
        kt = k[:, t].repeat_interleave(rep, 1).unsqueeze(-1)
        qt = q[:, t].repeat_interleave(rep, 1).unsqueeze(-1)
        St = St * dec[:, t, :, None, None]
        d = (v[:, t] - (kt * St).sum(-2)) * beta[:, t].unsqueeze(-1)
        St = St + kt * d.unsqueeze(-2)
        o[:, t] = (qt * St).sum(-2)
    S[slot] = _pack(St).reshape(B, HV, DK * DV)
    o = _rnd(torch.cat([o[i, :n[i]] for i in range(B)]))
    x1 = _rnd(o / torch.sqrt(o.square().mean(-1, keepdim=True) + EPS))
    x2 = _rnd(x1 * w["onorm_w"].double())
    zz = z.reshape(-1, HV, DV)
    return (x2 * (zz * _sig(zz))).reshape(-1, VD), conv, S


def _rope_norm(x, w, pos):
    """(1+w) RMSNorm, then rotary dims; x [T, h, D] float64, pos [T]."""
    x = _rnd(x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + w.double()))
    h = ROT // 2
    inv = torch.tensor([THETA ** (-2.0 * i / ROT) for i in range(h)], dtype=torch.float64)
    # the angle is a float32 product by definition
    ang = (pos.float().unsqueeze(-1) * inv.float().to("cuda")).double().unsqueeze(1)
    c, sn = _rnd(torch.cos(ang)), _rnd(torch.sin(ang))
    lo, hi = x[..., :h], x[..., h:ROT]
    return torch.cat([_rnd(_rnd(lo * c) + _rnd(-hi * sn)), _rnd(_rnd(hi * c) + _rnd(lo * sn)),
                      x[..., ROT:]], -1)


def _exact_attn(s, qg, k, v):
    """(y, k_cache, v_cache) of the GQA mixer for float64 inputs."""
    w, n, ctx, cu = s["w"], s["new"], s["ctx"], s["cu"]
    kc, vc = s["k_cache"].clone(), s["v_cache"].clone()
    out = torch.empty(int(cu[-1]), NH, D, device="cuda", dtype=torch.float64)
    for i in range(len(n)):
        r = slice(int(cu[i]), int(cu[i + 1]))
        pos = torch.arange(ctx[i], ctx[i] + n[i], device="cuda")
        q = _rope_norm(qg[r, :, :D], w["qn_w"], pos)
        ids = torch.from_numpy(s["table"][i].astype(np.int64)).to("cuda")[pos // BLK]
        kc[ids, :, pos % BLK] = _rope_norm(k[r], w["kn_w"], pos).to(BF)
        vc[ids, :, :, pos % BLK] = v[r].to(BF)
        used = torch.from_numpy(s["table"][i, :s["nblk"][i]].astype(np.int64)).to("cuda")
        last = ctx[i] + n[i]
        hidden = torch.arange(last, device="cuda").unsqueeze(0) > pos.unsqueeze(1)
        for g in range(NKV):
            K = kc[used, g].reshape(-1, D)[:last].double()
            V = vc[used, g].transpose(1, 2).reshape(-1, D)[:last].double()
            for h in range(g * GRP, (g + 1) * GRP):
                A = _rnd(_rnd(q[:, h].contiguous() @ K.t().contiguous()) * D ** -0.5)
                A.masked_fill_(hidden, -math.inf)
                P = _rnd(torch.softmax(A, -1))
                out[r, h] = _rnd(P @ V)
    y = out * _rnd(_sig(qg[..., D:]))
    return y.reshape(-1, NH * D), kc, vc


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "proj":
        return {"y": s["x"].double() @ s["wt"].double().t().contiguous()}
    x = s["ln1"].double() if case["kind"] == "layer" else None

    def proj(name):
        return _rnd(x @ s["pw"][name].double().t().contiguous())
    if _mixer(case) == "gdn":
        if case["kind"] == "layer":
            y, conv, S = _exact_gdn(s, proj("w_qkv"), proj("w_z"), proj("w_a"), proj("w_b"))
            y = _rnd(y) @ s["pw"]["w_out"].double().t().contiguous()
        else:
            y, conv, S = _exact_gdn(s, *(s[f].double() for f in ("qkv", "z", "a", "b")))
        return {"y": y, "conv": conv, "S": S}
    if case["kind"] == "layer":
        y, kc, vc = _exact_attn(s, proj("wq").reshape(-1, NH, 2 * D),
                                proj("wk").reshape(-1, NKV, D), proj("wv").reshape(-1, NKV, D))
        y = _rnd(y) @ s["pw"]["wo"].double().t().contiguous()
    else:
        y, kc, vc = _exact_attn(s, *(s[f].double() for f in ("qg", "k", "v")))
    return {"y": y, "k_cache": kc, "v_cache": vc}
