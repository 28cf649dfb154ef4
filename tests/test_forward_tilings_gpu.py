"""The tilings that small forwards take by the cost estimate (8 steps a lane, twelve waves), at lengths around the
edges of their slices and chunks: bit for bit the sequential model of the composition order, and the
gated scan that of the plain scan on the alpha and beta it forms."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from fast_sequential_scan_amd import _native  # noqa: E402
from fast_sequential_scan_amd import sequential_scan_cuda as ext  # noqa: E402
from fast_sequential_scan_amd.workloads import make_inputs  # noqa: E402

DEV = "cuda:0"
CODE = {torch.bfloat16: _native.FSS_BF16, torch.float32: _native.FSS_F32}


def plan(shape, dtype, direction):
    out = (ctypes.c_int32 * 8)()
    assert _native.lib().fss_debug_chain_plan(*shape, CODE[dtype], direction, 16, None, out) == 0
    n_chunks, waves, steps, period, look, span, _vec, _cols = list(out)
    return dict(steps=steps, waves=waves, period=period, look=look, span=span)


def bits(t):
    t = t.detach().cpu().contiguous()
    return t.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.numpy()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [
    (1, 65, 64), (3, 127, 70), (3, 128, 72), (2, 129, 200), (1, 697, 448), (5, 511, 131), (5, 513, 129), (24, 766, 512),
    (24, 769, 512), (10, 1728, 256), (10, 1729, 256), (10, 1919, 250), (1, 40000, 65)])
def test_forward_is_the_model_bit_for_bit(oracle, dtype, shape):
    alpha, beta, _ = make_inputs("near_one", *shape, dtype=dtype, seed=sum(shape))
    a, b = alpha.to(DEV), beta.to(DEV)
    got = ext._forward(dtype, a, b)
    want = oracle.chained_scan_fwd(bits(alpha), bits(beta), **plan(shape, dtype, _native.FSS_FWD))
    ext.workspace_status()
    assert np.array_equal(bits(got).view(np.uint16 if dtype == torch.bfloat16 else np.uint32),
                          want.view(np.uint16 if dtype == torch.bfloat16 else np.uint32))
    # with a state coming in and going out the sequence is cut at the same places: a zero state changes no bit
    zero = torch.zeros(shape[0], shape[2], device=DEV)
    h, last = ext.scan_forward_state(a, b, zero)
    assert torch.equal(h, got) and torch.equal(last.to(dtype), got[:, -1])


# the last six: the tilings of launches that fill the device, short and odd and long
@pytest.mark.parametrize("shape,dtype", [
    ((2, 65, 130), torch.bfloat16), ((3, 614, 1006), torch.bfloat16), ((10, 1871, 256), torch.bfloat16), ((10, 1727, 256), torch.bfloat16),
    ((10, 1920, 252), torch.bfloat16), ((7, 300, 513), torch.bfloat16),
    ((29, 299, 1000), torch.bfloat16), ((33, 512, 512), torch.bfloat16), ((9, 1800, 519), torch.bfloat16), ((1, 16400, 520), torch.bfloat16),
    ((2, 2500, 1700), torch.bfloat16), ((3, 1500, 1000), torch.float32)])
def test_gated_forward_matches_oracle(oracle, shape, dtype):
    g = torch.Generator().manual_seed(sum(shape))
    gate = (1.5 * torch.randn(shape, generator=g)).to(dtype)
    x = torch.randn(shape, generator=g).to(dtype)
    got = ext.gated_scan_forward(gate.to(DEV), x.to(DEV)).float().cpu().numpy()
    ext.workspace_status()
    rounding, rtol, atol = ("bf16", 1e-2, 1e-2) if dtype == torch.bfloat16 else ("f32", 1e-4, 1e-5)  # (the bars of tests/test_scan_gated_gpu.py)
    g32, x32 = gate.float().numpy(), x.float().numpy()
    # (from either rounding of an alpha that lies on the edge of one)
    ok = oracle.within_rounding_envelope(got, oracle.gated_scan_fwd(g32, x32, rounding), oracle.gated_scan_fwd(g32, x32, rounding, True),
                                         rtol, atol)
    assert ok.all(), (~ok).sum()
