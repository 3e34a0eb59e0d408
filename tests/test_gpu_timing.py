"""The timing hook (apus_hip_timing_get) reports each launch under the name
of the kernel that ran, where a call's sizes choose between kernels."""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


def _td(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to("cuda")


def _launches(hip, call, *names):
    hip.timing_enable(True)
    try:
        call()
        return [hip.timing_get(n)[1] for n in names]
    finally:
        hip.timing_enable(False)


@pytest.mark.parametrize("M,O,K,exact,ran,other", [
    (16, 512, 64, False, "k_gemm_tile", "k_gemm_wide"),
    (2048, 2048, 64, False, "k_gemm_wide", "k_gemm_tile"),
    (2, 128, 128, True, "k_gemm_seq64", "k_gemm_seq"),
    (2, 128, 40, True, "k_gemm_seq", "k_gemm_seq64")])
def test_timing_names_gemm(hip, M, O, K, exact, ran, other):
    import torch
    w, x, y = (torch.zeros(s, dtype=torch.int16, device="cuda") for s in ((O, K), (M, K), (M, O)))
    assert _launches(hip, lambda: hip.bf16_gemm_dev(w, x, y, exact=exact), ran, other) == [1, 0]


@pytest.mark.parametrize("T,ran,other", [(64, "k_attn_fa16", "k_attn_fa"),
                                         (8192, "k_attn_fa", "k_attn_fa16")])
def test_timing_names_prefill(hip, T, ran, other):
    import torch
    dims = synth.ATTN_DIMS
    nh, nkv, d = dims[:3]
    rng = np.random.default_rng(T)
    layer = hip.attn_layer(dims, {k: _td(torch, v) for k, v in synth.attn_weights(rng).items()})
    z = lambda *s: torch.zeros(s, dtype=torch.int16, device="cuda")
    qg, k, v, y = z(T, nh, 2 * d), z(T, nkv, d), z(T, nkv, d), z(T, nh * d)
    dk, dv = z(1, nkv, T, d), z(1, nkv, T // 32, d, 32)
    call = lambda: hip.attn_prefill(layer, [0, T], [0], qg, k, v, dk, dv, T, y)
    assert _launches(hip, call, ran, other) == [1, 0]


@pytest.mark.parametrize("B,ran,other", [(1, "k_attn_scores_few", "k_attn_scores"),
                                         (40, "k_attn_scores", "k_attn_scores_few")])
def test_timing_names_decode(hip, B, ran, other):
    """126 64-key groups per sequence and kv head; k_attn_scores_few takes
    calls of up to 8192 of them."""
    import torch
    dims = synth.ATTN_DIMS
    nh, nkv, d = dims[:3]
    pos, max_seq = 8000, 8032
    rng = np.random.default_rng(B)
    layer = hip.attn_layer(dims, {k: _td(torch, v) for k, v in synth.attn_weights(rng).items()})
    z = lambda *s: torch.zeros(s, dtype=torch.int16, device="cuda")
    qg, k, v, y = z(B, nh, 2 * d), z(B, nkv, d), z(B, nkv, d), z(B, nh * d)
    dk, dv = z(B, nkv, max_seq, d), z(B, nkv, max_seq // 32, d, 32)
    call = lambda: hip.attn_decode(layer, np.arange(B + 1), np.full(B, pos), qg, k, v, dk, dv,
                                   max_seq, y)
    assert _launches(hip, call, ran, other) == [1, 0]
