"""GPU parity: chunked GDN prefill (apus_hip_gdn_prefill) against the
oracle's sequential recurrence.

The chunk (WY/UT) form sums in a different order from the reference's
token loop (c/gdn.h:627-635), so it is a tolerance class of it:
  * recurrent state: max |S - S_ref| / max |S_ref| <= 1e-4;
  * y (after rnd(o) and the three-rounding gated RMSNorm): normwise
    relative error <= 2e-3 and at most 4 bf16 ulps per element (an fp32
    ulp of o that crosses a bf16 rounding boundary moves rnd(o) by one
    ulp and each of the norm's three roundings by at most one more),
    elements small through cancellation judged against their row's rms
    (numerics.assert_bf16_rows);
  * conv state: bit-exact (pure copies of input codes).
Cases: ragged batches with partial chunks (1, 63, 64, 65, 130 tokens) from
a prior state, BASELINE config 1 (T=4096 from zero state), and a strong
decay case where cumulative in-chunk decay underflows fp32.
"""
import numpy as np
import pytest

import synth
from numerics import assert_bf16_close, assert_bf16_rows, assert_state_close

pytestmark = pytest.mark.gpu


def _dev(torch, arr):
    return torch.from_numpy(arr.view(np.int16) if arr.dtype == np.uint16 else arr).to("cuda")


def _run_prefill(hip, orc, rng, cu, zero_state=False, a_scale=1.0, tag=""):
    import torch
    dims = synth.GDN_DIMS
    B = len(cu) - 1
    T = int(cu[-1])
    w = synth.gdn_weights(rng)
    tok = synth.gdn_tokens(rng, T)
    if a_scale != 1.0:
        tok["a"] = synth.bf16_bits(synth.bf16_f32(tok["a"]) * np.float32(a_scale) + np.float32(4.0))
    conv, S = synth.gdn_state(rng, B, zero=zero_state)
    print(f"[gdn_prefill {tag}] B={B} T={T} cu={list(cu)[:8]}...", flush=True)
    c_o, S_o = conv.copy(), S.copy()
    y_o = orc.gdn_mixer(dims, w, np.asarray(cu, np.int32), tok["qkv"], tok["z"], tok["a"],
                        tok["b"], c_o, S_o)
    tw = {k: _dev(torch, v) for k, v in w.items()}
    layer = hip.gdn_layer(dims, tw)
    t = {k: _dev(torch, v) for k, v in tok.items()}
    dconv = _dev(torch, conv)
    dS_ref = torch.from_numpy(S).cuda()
    dS = torch.empty_like(dS_ref)
    hip.gdn_state_pack(dS_ref, dS)
    y = torch.empty((T, dims[1] * dims[3]), dtype=torch.int16, device="cuda")
    hip.gdn_prefill(layer, cu, t["qkv"], t["z"], t["a"], t["b"], dconv, dS, y)
    hip.gdn_state_unpack(dS, dS_ref)
    torch.cuda.synchronize()
    y_h = y.cpu().numpy().view(np.uint16)
    assert np.array_equal(dconv.cpu().numpy().view(np.uint16), c_o), "conv state"
    e = assert_state_close(dS_ref.cpu().numpy(), S_o, what=f"prefill S {tag}")
    st = assert_bf16_rows(y_h, y_o, 128, what=f"prefill y {tag}")
    print(f"[gdn_prefill {tag}] y {st} state rel {e:.3g}", flush=True)
    return st, e


def test_prefill_ragged(hip, orc):
    """Partial and exact chunks, a one-token sequence, prior state."""
    lens = [1, 63, 64, 65, 130, 7]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    _run_prefill(hip, orc, np.random.default_rng(1001), cu, tag="ragged")


def test_prefill_config1(hip, orc):
    """batch 1, T=4096, zero initial state."""
    _run_prefill(hip, orc, np.random.default_rng(12), np.array([0, 4096], np.int32),
                 zero_state=True, tag="config1")


def test_prefill_strong_decay(hip, orc):
    """a shifted up by 4 (softplus ~ 4-8 per token, with A_log up to 2.7 the
    log decay reaches -100 per token): exp(gamma) of a chunk underflows and
    the state forgets within a few tokens."""
    _run_prefill(hip, orc, np.random.default_rng(77), np.array([0, 200], np.int32),
                 a_scale=2.0, tag="strong_decay")


@pytest.mark.parametrize("swap", [False, True])
def test_prefill_silu_every_code(hip, orc, swap):
    """The chunk kernel's SiLU (from the table for one channel of a pair, by
    formula with the table behind it for the other) on every bf16 code of
    magnitude 2^-80 .. 2^40 above -64 (below it the product goes to 0): 16
    one-token sequences from a zero state, whose conv passes the codes
    through (last tap 1); swap: with the two channels of every pair
    exchanged, so that over both runs each code takes either way. S = beta k
    v^T then, so column j shows v_j = SiLU(code) to the chunk form's own
    1e-5, against 2^-8 for a code that is one ulp off."""
    import torch
    dims = synth.GDN_DIMS
    hk, hv, dk, dv = dims
    rng = np.random.default_rng(8)
    B, cd, kd = 16, 2 * hk * dk + hv * dv, hk * dk
    w = synth.gdn_weights(rng)
    w["conv_w"] = np.zeros((cd, 4), np.uint16)
    w["conv_w"][:, 3] = 0x3F80
    tok = synth.gdn_tokens(rng, B)
    codes = rng.permutation(np.arange(1 << 16, dtype=np.uint32)).astype(np.uint16)
    exp = (codes >> 7) & 0xFF
    codes = np.where((exp >= 127 - 80) & (exp <= np.where(codes >> 15, 127 + 5, 127 + 40)), codes,
                     0x3F80)
    if swap:
        codes = np.ascontiguousarray(codes.reshape(-1, 2)[:, ::-1])
    tok["qkv"][:, 2 * kd:] = codes.reshape(B, hv * dv)
    conv, S = synth.gdn_state(rng, B, zero=True)
    cu = np.arange(B + 1, dtype=np.int32)
    S_o = S.copy()
    orc.gdn_mixer(dims, w, cu, tok["qkv"], tok["z"], tok["a"], tok["b"], conv.copy(), S_o)
    layer = hip.gdn_layer(dims, {k: _dev(torch, v) for k, v in w.items()})
    t = {k: _dev(torch, v) for k, v in tok.items()}
    dS = torch.zeros((B, hv, dk, dv), device="cuda")
    out = torch.empty_like(dS)
    y = torch.empty((B, hv * dv), dtype=torch.int16, device="cuda")
    hip.gdn_prefill(layer, cu, t["qkv"], t["z"], t["a"], t["b"], _dev(torch, conv), dS, y)
    hip.gdn_state_unpack(dS, out)
    torch.cuda.synchronize()
    r = S_o.astype(np.float64)
    err = np.abs(out.cpu().numpy() - r).max(axis=2) / np.abs(r).max(axis=2)
    assert err.max() <= 1e-4, float(err.max())


def test_prefill_conv_small_products(hip, orc):
    """The conv's products are rounded before they are added, as the
    reference's are, also below 2^-126, where the product of two bf16 values
    is not exact in fp32. Every v channel's taps give, with u = 2^-149,
    32767 u, 1.5 u, 2^-110 and 2^-118: with 1.5 u rounded to 2 u first the
    first two pass half an ulp of 2^-110, the sum lies above a bf16 tie and
    the code is 2^-110 (1 + 2^-7); added unrounded they make 32768 u, both
    ties go to even and the code is 2^-110. One token from a zero state, so
    S = beta k v^T shows v to the chunk form's own 1e-5 against 2^-7."""
    import torch
    dims = synth.GDN_DIMS
    hk, hv, dk, dv = dims
    rng = np.random.default_rng(9)
    kd = hk * dk
    w = synth.gdn_weights(rng)
    tok = synth.gdn_tokens(rng, 1)
    conv, S = synth.gdn_state(rng, 1, zero=True)
    taps = np.array([217.0, 3.0, 1.0, 1.0]) * np.exp2([-75.0, -75.0, -55.0, -59.0])
    vals = np.array([151.0, 1.0, 1.0, 1.0]) * np.exp2([-74.0, -75.0, -55.0, -59.0])
    w["conv_w"] = w["conv_w"].copy()
    w["conv_w"].reshape(-1, 4)[2 * kd:] = synth.bf16_bits(taps.astype(np.float32))
    x = synth.bf16_bits(vals.astype(np.float32))
    conv.reshape(-1, 3)[2 * kd:] = x[:3]
    tok["qkv"].reshape(-1)[2 * kd:] = x[3]
    cu = np.array([0, 1], np.int32)
    S_o = S.copy()
    orc.gdn_mixer(dims, w, cu, tok["qkv"], tok["z"], tok["a"], tok["b"], conv.copy(), S_o)
    layer = hip.gdn_layer(dims, {k: _dev(torch, v) for k, v in w.items()})
    t = {k: _dev(torch, v) for k, v in tok.items()}
    dS = torch.zeros((1, hv, dk, dv), device="cuda")
    out = torch.empty_like(dS)
    y = torch.empty((1, hv * dv), dtype=torch.int16, device="cuda")
    hip.gdn_prefill(layer, cu, t["qkv"], t["z"], t["a"], t["b"], _dev(torch, conv), dS, y)
    hip.gdn_state_unpack(dS, out)
    torch.cuda.synchronize()
    r = S_o.astype(np.float64)
    assert np.abs(r).max() > 0.0
    err = np.abs(out.cpu().numpy() - r).max(axis=2) / np.abs(r).max(axis=2)
    assert err.max() <= 1e-4, float(err.max())


def test_prefill_then_decode(hip, orc):
    """Prefill a prompt then decode one token from the device state: the
    state layout and conv state the prefill leaves are what decode reads."""
    import torch
    dims = synth.GDN_DIMS
    rng = np.random.default_rng(31)
    T = 100
    w = synth.gdn_weights(rng)
    tok = synth.gdn_tokens(rng, T + 1)
    conv, S = synth.gdn_state(rng, 1, zero=True)
    c_o, S_o = conv.copy(), S.copy()
    y_o = orc.gdn_mixer(dims, w, np.array([0, T + 1], np.int32), tok["qkv"], tok["z"], tok["a"],
                        tok["b"], c_o, S_o)
    tw = {k: _dev(torch, v) for k, v in w.items()}
    layer = hip.gdn_layer(dims, tw)
    t = {k: _dev(torch, v) for k, v in tok.items()}
    dconv = _dev(torch, conv)
    dS = torch.zeros(S.shape, dtype=torch.float32, device="cuda")
    y = torch.empty((T + 1, dims[1] * dims[3]), dtype=torch.int16, device="cuda")
    hip.gdn_prefill(layer, [0, T], t["qkv"][:T], t["z"][:T], t["a"][:T], t["b"][:T], dconv, dS,
                    y[:T])
    hip.gdn_decode(layer, [0, 1], t["qkv"][T:], t["z"][T:], t["a"][T:], t["b"][T:], dconv, dS,
                   y[T:])
    Su = torch.empty_like(dS)
    hip.gdn_state_unpack(dS, Su)
    torch.cuda.synchronize()
    assert np.array_equal(dconv.cpu().numpy().view(np.uint16), c_o)
    assert_state_close(Su.cpu().numpy(), S_o, what="prefill+decode S")
    assert_bf16_rows(y.cpu().numpy().view(np.uint16), y_o, 128, what="prefill+decode y")


@pytest.mark.parametrize("B", [260, 410])
def test_prefill_many_sequences(hip, orc, B):
    """Batches past the by-value metadata limits (256 sequences for the
    token-parallel kernels, 400 for the chunk kernels): the offsets then
    travel through a device copy."""
    rng = np.random.default_rng(B)
    lens = rng.integers(1, 5, B)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    _run_prefill(hip, orc, rng, cu, tag=f"B{B}")


def test_prefill_batched_equals_alone(hip):
    """The reference's batch invariance (batched prefill == sequential,
    bitwise; tests/m9c): a ragged batch of 5 sequences and each sequence
    prefilled alone give the same outputs, conv state and recurrent state,
    bit for bit (a sequence's chunks start at its own first token either
    way)."""
    import torch
    rng = np.random.default_rng(95)
    dims = synth.GDN_DIMS
    k = [1, 63, 64, 65, 130]
    cu = np.concatenate([[0], np.cumsum(k)]).astype(np.int32)
    B, T = len(k), int(cu[-1])
    w = synth.gdn_weights(rng)
    tok = synth.gdn_tokens(rng, T)
    conv, S = synth.gdn_state(rng, B)
    layer = hip.gdn_layer(dims, {n: _dev(torch, v) for n, v in w.items()})
    t = {n: _dev(torch, v) for n, v in tok.items()}
    dS0 = torch.empty((B,) + S.shape[1:], dtype=torch.float32, device="cuda")
    hip.gdn_state_pack(torch.from_numpy(S).cuda(), dS0)
    vd = dims[1] * dims[3]
    c1, S1 = _dev(torch, conv), dS0.clone()
    y1 = torch.empty((T, vd), dtype=torch.int16, device="cuda")
    hip.gdn_prefill(layer, cu, t["qkv"], t["z"], t["a"], t["b"], c1, S1, y1)
    c2, S2 = _dev(torch, conv), dS0.clone()
    y2 = torch.empty((T, vd), dtype=torch.int16, device="cuda")
    for s in range(B):
        a, b = int(cu[s]), int(cu[s + 1])
        hip.gdn_prefill(layer, [0, b - a], t["qkv"][a:b], t["z"][a:b], t["a"][a:b], t["b"][a:b],
                        c2[s:s + 1], S2[s:s + 1], y2[a:b])
    torch.cuda.synchronize()
    assert torch.equal(y1, y2), "outputs"
    assert torch.equal(c1, c2), "conv state"
    assert torch.equal(S1, S2), "recurrent state"
