"""GPU parity: the projections on either side of the path (c/bf16.h:
178-231) through the C ABI against the oracle (itself bitwise the
reference's x86 hot path, tests/test_oracle_ref.py).

The hook drop-ins (host pointers) and the device-pointer sequential kernel
keep the reference's order and must be bitwise. The MFMA GEMM (hand-written,
every row count) sums in the MFMA's order: every element within 2e-3 (|r| + esc), esc = sum_k |w x|
(the attention kernels' class), and normwise within 2e-3.
"""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu

SHAPES = [(1, 12352, 2048),     # GDN in_proj (qkv | z | a | b) at one token
          (3, 2048, 4096),      # GDN out_proj, three tokens
          (2, 517, 40),         # ragged outputs, a short K
          (1, 33, 37)]          # K not a multiple of 8 (the scalar path)


def _dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to("cuda")


@pytest.mark.parametrize("M,O,K", SHAPES)
def test_gemm_hooks_bitwise(hip, orc, M, O, K):
    rng = np.random.default_rng(M * 1000003 + O * 7 + K)
    w = synth.normal_bf16(rng, (O, K), K ** -0.5)
    x = synth.normal_bf16(rng, (M, K))
    print(f"[proj] hooks M={M} O={O} K={K}", flush=True)
    y = hip.bf16_gemm(w, x)
    r = orc.bf16_gemm(w, x)
    assert np.array_equal(y, r)
    assert np.array_equal(hip.bf16_gemv(w, np.ascontiguousarray(x[0])), r[0])


def test_gemm_hooks_weight_copies(hip, orc):
    """Weights are copied once per host buffer: repeated calls reuse the
    copy; another buffer (or a released cache) gets its own."""
    rng = np.random.default_rng(5)
    w1 = synth.normal_bf16(rng, (300, 256), 0.1)
    w2 = synth.normal_bf16(rng, (300, 256), 0.1)
    x = synth.normal_bf16(rng, (2, 256))
    for _ in range(2):
        assert np.array_equal(hip.bf16_gemm(w1, x), orc.bf16_gemm(w1, x))
        assert np.array_equal(hip.bf16_gemm(w2, x), orc.bf16_gemm(w2, x))
    hip.bf16_weights_release()
    w1[:] = w2
    assert np.array_equal(hip.bf16_gemm(w1, x), orc.bf16_gemm(w2, x))


@pytest.mark.parametrize("M,O,K", SHAPES)
def test_gemm_dev_bitwise(hip, orc, M, O, K):
    import torch
    rng = np.random.default_rng(M + O + K)
    w = synth.normal_bf16(rng, (O, K), K ** -0.5)
    x = synth.normal_bf16(rng, (M, K))
    y = torch.empty((M, O), dtype=torch.int16, device="cuda")
    hip.bf16_gemm_dev(_dev(torch, w), _dev(torch, x), y, exact=True)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), orc.bf16_gemm(w, x))


# K a multiple of 64 (weights streamed by wavefronts of their own): one
# chunk, fewer chunks than are kept in flight, one more; one to four rows a
# workgroup with a remainder; outputs past a workgroup's 64; the largest K
@pytest.mark.parametrize("M,O,K", [(1, 64, 64), (5, 70, 128), (3, 4100, 576), (2, 65, 16384),
                                   (7, 12352, 512), (11, 8200, 192), (1, 130, 16448)])
def test_gemm_dev_bitwise_chunks(hip, orc, M, O, K):
    import torch
    rng = np.random.default_rng(M * O + K)
    w = synth.normal_bf16(rng, (O, K), K ** -0.5)
    x = synth.normal_bf16(rng, (M, K))
    print(f"[proj] chunks M={M} O={O} K={K}", flush=True)
    y = torch.empty((M, O), dtype=torch.int16, device="cuda")
    hip.bf16_gemm_dev(_dev(torch, w), _dev(torch, x), y, exact=True)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), orc.bf16_gemm(w, x))


@pytest.mark.parametrize("M,O", [(1, 1), (1, 130), (5, 64)])
def test_gemm_empty_sums(hip, M, O):
    """K = 0: every output is an empty sum, +0, and no operand is read."""
    import torch
    w, x = (torch.empty((n, 0), dtype=torch.int16, device="cuda") for n in (O, M))
    y = torch.full((M, O), -1, dtype=torch.int16, device="cuda")
    print(f"[proj] empty sums M={M} O={O}", flush=True)
    hip.bf16_gemm_dev(w, x, y, exact=True)
    torch.cuda.synchronize()
    assert not y.cpu().any()
    assert not hip.bf16_gemm(np.empty((O, 0), np.uint16), np.empty((M, 0), np.uint16)).any()


def test_gemm_dev_bitwise_wide_range(hip, orc):
    """Operands whose magnitudes span 2^-60 .. 2^60 (every product still in
    fp32's normal range): the sequential kernel's fused multiply-add rounds
    where the reference's multiply-then-add does, so the result stays
    bitwise; exact zeros and sign mixes included."""
    import torch
    rng = np.random.default_rng(77)
    O, K, M = 4096, 2048, 2
    def wide(shape):
        v = rng.standard_normal(shape) * np.exp2(rng.integers(-60, 61, shape))
        v[rng.random(shape) < 0.05] = 0.0
        return synth.bf16_bits(v.astype(np.float32))
    w, x = wide((O, K)), wide((M, K))
    y = torch.empty((M, O), dtype=torch.int16, device="cuda")
    hip.bf16_gemm_dev(_dev(torch, w), _dev(torch, x), y, exact=True)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint16), orc.bf16_gemm(w, x))
    assert np.array_equal(hip.bf16_gemv(w, np.ascontiguousarray(x[0])), orc.bf16_gemm(w, x)[0])


# from one tile to most of a chip of them, with ragged row / output
# edges, a split K, and an output count that is not a multiple of 4 (the
# element-store epilogue)
@pytest.mark.parametrize("M,O,K", [(64, 12352, 2048), (200, 1000, 4096), (1, 70, 32),
                                   (300, 5000, 512),
                                   (260, 10240, 256),
                                   (1000, 1000, 512),   # ragged edges
                                   (700, 517, 64)])     # O % 4 != 0
def test_gemm_mfma_tolerance(hip, orc, M, O, K):
    import torch
    rng = np.random.default_rng(M * 31 + K)
    w = synth.normal_bf16(rng, (O, K), K ** -0.5)
    x = synth.normal_bf16(rng, (M, K))
    print(f"[proj] mfma M={M} O={O} K={K}", flush=True)
    y = torch.empty((M, O), dtype=torch.int16, device="cuda")
    hip.bf16_gemm_dev(_dev(torch, w), _dev(torch, x), y, exact=False)
    torch.cuda.synchronize()
    c = synth.bf16_f32(y.cpu().numpy().view(np.uint16)).astype(np.float64)
    r = synth.bf16_f32(orc.bf16_gemm(w, x)).astype(np.float64)
    esc = np.abs(synth.bf16_f32(x).astype(np.float64)) @ np.abs(synth.bf16_f32(w).astype(np.float64)).T
    assert np.all(np.abs(c - r) <= 2e-3 * (np.abs(r) + esc))
    nrm = np.linalg.norm(c - r) / np.linalg.norm(r)
    same = float(np.mean(c == r))
    print(f"[proj] mfma normwise {nrm:.3g}, identical {same:.4f}", flush=True)
    assert nrm <= 2e-3 and same > 0.9


# The tile shape follows the call's size; an element's k16 steps are summed
# in the same order in all of them, so a call of many rows gives bit for bit
# what 64-row calls (the smallest tile) give. Row and output edges of the
# 128- to 256-wide tiles, a last output tile of at most 64 outputs and one of
# more, output counts that are not a multiple of 8 (element stores), K of one
# stage, of half a stage and with an odd half stage.
@pytest.mark.parametrize("M,O,K", [(4096, 576, 64), (2300, 4160, 2048), (1025, 12352, 96),
                                   (700, 12353, 32), (1537, 8200, 160), (769, 12356, 2080),
                                   (385, 12320, 64), (129, 12352, 192), (3001, 2049, 1056),
                                   (200, 12352, 32), (325, 12352, 128), (300, 12345, 288)])
def test_gemm_mfma_tile_shapes_agree(hip, M, O, K):
    import torch
    print(f"[proj] shapes M={M} O={O} K={K}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + O + K)
    w = (torch.randn(O, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    y = torch.zeros((M, O), dtype=torch.bfloat16, device="cuda")
    hip.bf16_gemm_dev(w, x, y, exact=False)
    part = torch.zeros_like(y)
    for m in range(0, M, 64):
        hip.bf16_gemm_dev(w, x[m:m + 64], part[m:m + 64], exact=False)
    assert torch.equal(y.view(torch.int16), part.view(torch.int16))
    r = x.double() @ w.double().t().contiguous()
    assert float((y.double() - r).norm() / r.norm()) <= 2e-3      # rnd alone: 1.7e-3


def test_gemm_mfma_refuses_unaligned_k(hip):
    """K not a multiple of 32: the MFMA GEMM returns "unsupported" (the
    caller runs the exact kernel or its CPU op), never a wrong result."""
    import torch
    w = torch.zeros((90, 40), dtype=torch.int16, device="cuda")
    x = torch.zeros((7, 40), dtype=torch.int16, device="cuda")
    y = torch.empty((7, 90), dtype=torch.int16, device="cuda")
    with pytest.raises(hip.ApusHipError) as e:
        hip.bf16_gemm_dev(w, x, y, exact=False)
    assert e.value.code == 1
