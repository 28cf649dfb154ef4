"""Rows that are no whole number of cache lines: column tiles meet on the lines at their seams, and the
kernels take their tiles in another order there (and, where the rows are no whole 64-byte sectors
either, without cache hints).  Against the oracle, under grids that cut their rounds at every offset;
which tile a workgroup takes must not show in the results, so all grids give the same bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from fast_sequential_scan_amd import sequential_scan_cuda as ext  # noqa: E402

DEV = "cuda:0"
TOL = {torch.bfloat16: (1e-2, 1e-2), torch.float16: (2e-3, 2e-3), torch.float32: (1e-4, 1e-5)}


def _check(got, want, dtype, what):
    rtol, atol = TOL[dtype]
    np.testing.assert_allclose(got.float().cpu().numpy(), want, rtol=rtol, atol=atol, err_msg=what)


# (bs, seq, d): rows of whole sectors (352 -> 704 bytes in 16 bits), of none (300, 1001), one tile per row (70),
# numbers of column groups that divide by 8 and that do not, chunks that fill the last round partly
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bs,seq,d", [(3, 700, 352), (2, 1030, 300), (1, 2049, 1001), (8, 130, 300), (5, 600, 70)])
def test_rows_that_share_lines(oracle, bs, seq, d, dtype):
    rng = torch.Generator().manual_seed(seq + d)
    alpha, beta, dout = (t.to(dtype) for t in (
        torch.sigmoid(torch.randn(bs, seq, d, generator=rng)), torch.randn(bs, seq, d, generator=rng), torch.randn(bs, seq, d, generator=rng)))
    h0 = torch.randn(bs, d, generator=rng).to(DEV)
    a, b, do = alpha.to(DEV), beta.to(DEV), dout.to(DEV)
    a32, b32, d32 = alpha.float().numpy(), beta.float().numpy(), dout.float().numpy()
    h = ext._forward(dtype, a, b)
    ga, gb = ext._backward(dtype, a, h, do)
    _check(h, oracle.scan_fwd_f32(a32, b32), dtype, "h")
    ga_or, gb_or = oracle.scan_bwd_f32(a32, h.float().cpu().numpy(), d32)
    _check(ga, ga_or, dtype, "grad_alpha")
    _check(gb, gb_or, dtype, "grad_beta")
    vec = 2 if d % 2 == 0 and dtype != torch.float32 else 1
    for steps in (8, 16):
        results = []
        for groups in (0, 3, 17, 44):
            cfg = (vec, steps, 2, groups)
            results.append([ext._forward(dtype, a, b, cfg), *ext._backward(dtype, a, h, do, cfg),
                            *ext.scan_forward_state(a, b, h0, cfg), *ext.scan_backward_state(a, h, do, h0, h0, cfg),
                            ext.gated_scan_forward(b, do, (vec if dtype != torch.float32 else 1, steps, 2, groups)),
                            *ext.gated_scan_backward(b, do, h, do, (vec if dtype != torch.float32 else 1, steps, 2, groups))])
        _check(results[0][0], oracle.scan_fwd_f32(a32, b32), dtype, f"h, {steps} steps")
        for other in results[1:]:
            assert all(torch.equal(x, y) for x, y in zip(results[0], other))
    ext.workspace_status()
