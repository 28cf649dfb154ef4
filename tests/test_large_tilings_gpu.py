"""The tilings that large launches of odd, ragged and narrow rows take, through the library's own choice: bit for
bit the sequential model of the composition order, with states against the oracle on a sequence one step longer."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from fast_sequential_scan_amd import _native  # noqa: E402
from fast_sequential_scan_amd import sequential_scan_cuda as ext  # noqa: E402
from fast_sequential_scan_amd.workloads import make_inputs  # noqa: E402

DEV = "cuda:0"
FWD, BWD, GATED_FWD = _native.FSS_FWD, _native.FSS_BWD, _native.FSS_GATED_FWD
CODE = {torch.bfloat16: _native.FSS_BF16, torch.float32: _native.FSS_F32}


def plan(shape, dtype, direction, tiling):
    """The chain's plan, of the tiling (vec, steps, waves) that the case stands for."""
    out = (ctypes.c_int32 * 8)()
    assert _native.lib().fss_debug_chain_plan(*shape, CODE[dtype], direction, 16, None, out) == 0
    _chunks, waves, steps, period, look, span, vec, cols = list(out)
    assert (vec, steps, waves * cols) == tiling, (shape, list(out))
    return dict(steps=steps, waves=waves, period=period, look=look, span=span)


def bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


@pytest.mark.parametrize("shape,fwd,bwd", [
    ((27, 6000, 210), (2, 32, 8), (2, 16, 12)),   # sector-sharing rows: 12 waves in the backward
    ((33, 1030, 990), (2, 32, 8), (2, 16, 12)),
    ((7, 4958, 969), (1, 32, 8), (1, 16, 16)),    # odd width: 16 waves in the backward
    ((24, 384, 1735), (1, 16, 8), (1, 16, 8)),     # odd width, short: 128-step chunks in the forward
    ((8, 11000, 192), (1, 32, 8), (1, 16, 16))])   # three column tiles: one channel per lane
def test_large_launches_are_the_model_bit_for_bit(oracle, shape, fwd, bwd):
    dtype = torch.bfloat16
    alpha, beta, dout = make_inputs("near_one", *shape, seed=sum(shape))
    a, b, do = alpha.to(DEV), beta.to(DEV), dout.to(DEV)
    h = ext._forward(dtype, a, b)
    ga, gb = ext._backward(dtype, a, h, do)
    ext.workspace_status()
    h_bits = bits(h)
    assert np.array_equal(h_bits, oracle.chained_scan_fwd(bits(alpha), bits(beta), **plan(shape, dtype, FWD, fwd)))
    ga_model, gb_model = oracle.chained_scan_bwd(bits(alpha), h_bits, bits(dout), **plan(shape, dtype, BWD, bwd))
    assert np.array_equal(bits(gb), gb_model)
    assert np.array_equal(bits(ga), ga_model)


@pytest.mark.parametrize("shape,tiling", [
    ((27, 6000, 210), (2, 16, 12)), ((7, 4958, 969), (1, 16, 16)), ((4, 11000, 192), (1, 16, 16))])
def test_large_backwards_with_states(oracle, shape, tiling):
    bs, seq, d = shape
    plan(shape, torch.bfloat16, BWD, tiling)
    alpha, beta, dout = make_inputs("sigmoid", *shape, seed=3)
    g = torch.Generator().manual_seed(4)
    h0, g_last = torch.randn(bs, d, generator=g), torch.randn(bs, d, generator=g)
    a, do = alpha.to(DEV), dout.to(DEV)
    h, h_last = ext.scan_forward_state(a, beta.to(DEV), h0.to(DEV))
    got = [h, h_last, *ext.scan_backward_state(a, h, do, h0.to(DEV), g_last.to(DEV))]
    ext.workspace_status()
    zeros = np.zeros((bs, 1, d), np.float32)
    a_ext = np.concatenate([zeros, alpha.float().numpy()], axis=1)
    h_ext = oracle.scan_fwd_f32(a_ext, np.concatenate([h0.numpy()[:, None], beta.float().numpy()], axis=1))
    d_ext = np.concatenate([zeros, dout.float().numpy()], axis=1)
    d_ext[:, -1] += g_last.numpy()
    ga_ext, gb_ext = oracle.scan_bwd_f32(a_ext, h_ext, d_ext)
    # (the bars of tests/test_scan_state_gpu.py)
    for name, x, want in zip(("h", "h_last", "grad_alpha", "grad_beta", "grad_h_before"), got,
                             (h_ext[:, 1:], h_ext[:, -1], ga_ext[:, 1:], gb_ext[:, 1:], gb_ext[:, 0])):
        x = x.float().cpu().numpy()
        assert (np.abs(x - want) <= 1e-2 + 1e-2 * np.abs(want)).all(), name


@pytest.mark.parametrize("shape,dtype,tiling", [
    ((34, 214, 664), torch.float32, (1, 16, 8)), ((24, 55, 3756), torch.float32, (1, 16, 4)),
    ((43, 32, 3345), torch.float32, (1, 16, 2)), ((9, 7795, 67), torch.float32, (1, 16, 12)),
    ((7, 5420, 175), torch.float32, (1, 16, 16)), ((2, 2048, 1024), torch.float32, (1, 16, 16)),
    ((4, 2048, 1024), torch.bfloat16, (2, 16, 16)), ((2, 4096, 1024), torch.bfloat16, (1, 32, 16)),
    ((11, 2100, 369), torch.bfloat16, (1, 16, 12)), ((64, 299, 440), torch.bfloat16, (2, 32, 16)), ((64, 299, 640), torch.bfloat16, (2, 16, 4))])
def test_large_gated_forwards(oracle, shape, dtype, tiling):
    plan(shape, dtype, GATED_FWD, tiling)
    g = torch.Generator().manual_seed(sum(shape))
    gate, x = ((s * torch.randn(shape, generator=g)).to(dtype) for s in (1.5, 1.0))
    got = ext.gated_scan_forward(gate.to(DEV), x.to(DEV)).float().cpu().numpy()
    ext.workspace_status()
    rounding, rtol, atol = ("bf16", 1e-2, 1e-2) if dtype == torch.bfloat16 else ("f32", 1e-4, 1e-5)  # (the bars of tests/test_scan_gated_gpu.py)
    g32, x32 = gate.float().numpy(), x.float().numpy()
    ok = oracle.within_rounding_envelope(got, oracle.gated_scan_fwd(g32, x32, rounding), oracle.gated_scan_fwd(g32, x32, rounding, True),
                                         rtol, atol)
    assert ok.all(), (~ok).sum()
