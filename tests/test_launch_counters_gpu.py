"""The launch number that tags a workspace's chaining words: every chained launch must move each of its
sixteen counters on by exactly one, whatever the grid, or words left by an earlier launch would
pass for valid ones."""
import ctypes

import pytest
import torch

from fast_sequential_scan_amd import _native
from fast_sequential_scan_amd import sequential_scan_cuda as ext
from fast_sequential_scan_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu

DEV = "cuda"
HEADER_BYTES, SLOT0_BYTES, SLOT_BYTES, SLOTS = 4096, 256, 128, 16


def counters(ws):
    words = ws[:HEADER_BYTES].view(torch.int64)
    return [int(words[(SLOT0_BYTES + s * SLOT_BYTES) // 8]) for s in range(SLOTS)]


@pytest.fixture(scope="module")
def case():
    alpha, beta, _ = make_inputs("near_one", 3, 1500, 200, seed=11)
    a, b = alpha.to(DEV), beta.to(DEV)
    return a, b


# grids below, at and above the number of counters (2 * 3 * 24 tiles of 8 steps and 8 waves), and uneven ones
@pytest.mark.parametrize("groups", [1, 2, 3, 7, 15, 16, 17, 31, 33, 100, 144])
def test_every_launch_moves_every_counter_on_by_one(case, groups):
    a, b = case
    lib = _native.lib()
    sp = torch.cuda.current_stream().cuda_stream
    cfg = _native.FssConfig(2, 8, 8, groups, 1)
    ws = torch.empty(lib.fss_workspace_bytes(*a.shape, _native.FSS_BF16, _native.FSS_FWD, ctypes.byref(cfg)),
                     dtype=torch.uint8, device=DEV)
    _native.check(lib.fss_workspace_init(ws.data_ptr(), ws.numel(), sp))
    want = ext._forward(torch.bfloat16, a, b, (2, 8, 8))

    def run(cfg=cfg):
        out = torch.full_like(a, float("nan"))
        _native.check(lib.fss_scan_fwd_ex(_native.FSS_BF16, a.data_ptr(), b.data_ptr(), out.data_ptr(), *a.shape,
                                          ws.data_ptr(), ws.numel(), sp, ctypes.byref(cfg)))
        return out

    for launch in range(1, 4):
        assert torch.equal(run(), want)
        assert counters(ws) == [launch << 32] * SLOTS
    # look-backs that are given up count like any other
    previous = lib.fss_debug_set_spin_limit(0)
    try:
        run()
        torch.cuda.synchronize()
    finally:
        lib.fss_debug_set_spin_limit(previous)
    assert counters(ws) == [4 << 32] * SLOTS
    # another grid on the same workspace, then this one again
    assert torch.equal(run(_native.FssConfig(2, 8, 8, 5, 1)), want)
    assert torch.equal(run(), want)
    assert counters(ws) == [6 << 32] * SLOTS


def test_the_number_wraps_without_the_tag_of_unwritten_words(case):
    a, b = case
    lib = _native.lib()
    sp = torch.cuda.current_stream().cuda_stream
    ws = torch.zeros(lib.fss_workspace_bytes_max(*a.shape), dtype=torch.uint8, device=DEV)
    words = ws[:HEADER_BYTES].view(torch.int64)
    for s in range(SLOTS):
        words[(SLOT0_BYTES + s * SLOT_BYTES) // 8] = -(2 << 32)  # two launches before the wrap
    want = ext.scan_forward_half(a, b)
    for _ in range(4):
        out = torch.empty_like(a)
        _native.check(lib.fss_scan_fwd_bf16(a.data_ptr(), b.data_ptr(), out.data_ptr(), *a.shape, ws.data_ptr(), ws.numel(), sp))
        assert torch.equal(out, want)
    assert counters(ws) == [2 << 32] * SLOTS


def test_row_major_and_channel_major_launches_share_a_workspace(case):
    a, b = case
    lib = _native.lib()
    sp = torch.cuda.current_stream().cuda_stream
    at, bt = (torch.cat([t.transpose(1, 2)] * 4, 2).contiguous() for t in (a, b))  # (3, 200, 6000): two chunks and more
    ws = torch.zeros(1 << 22, dtype=torch.uint8, device=DEV)
    want, want_cm = ext.scan_forward_half(a, b), ext.scan_forward_cm(at, bt)
    for launch in range(2):
        out, out_cm = torch.empty_like(a), torch.empty_like(at)
        _native.check(lib.fss_scan_fwd_bf16(a.data_ptr(), b.data_ptr(), out.data_ptr(), *a.shape, ws.data_ptr(), ws.numel(), sp))
        _native.check(lib.fss_scan_fwd_cm(_native.FSS_BF16, at.data_ptr(), bt.data_ptr(), out_cm.data_ptr(), *at.shape,
                                          ws.data_ptr(), ws.numel(), sp, None))
        assert torch.equal(out, want) and torch.equal(out_cm, want_cm)
    assert counters(ws) == [4 << 32] * SLOTS
