"""Host-side checks of how small forwards are tiled (the cost estimate in csrc/fss_host.h)."""
import csv
import ctypes
import os
import threading

import numpy as np
import pytest

from fast_sequential_scan_amd import _native

PAIRS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "forward_tilings_pairs.csv")
LIMIT = 4 << 20  # bytes of chaining words an estimate may ask for beyond the ladder's


def choose(lib, shape, dtype, direction, align=16):
    cfg = _native.FssConfig()
    assert lib.fss_choose_config(*shape, dtype, direction, align, ctypes.byref(cfg)) == 0
    return cfg.vec, cfg.steps, cfg.waves, cfg.cols


def test_chaining_words_stay_far_below_the_scratch_limits():
    """A tiling chosen by the estimate needs at most 4 MiB of words, or no more than the finest that launches that
    fill the device take (16 steps; 4 waves up to 2048 steps, 8 beyond).  In no case more than chunks of 64 steps would:
    24 bytes per chunk and channel, 6 % of what the forward moves in 16 bits.  (Not a promise that a workspace of one
    length serves every shorter one: see below.)"""
    lib = _native.lib()
    rng = np.random.default_rng(5)
    for _ in range(3000):
        d = int(rng.choice([1, 2, 3, 7, 63, 64, 65, 127, 200, 512, 1024]))
        bs = int(rng.choice([1, 2, 5, 64, 300]))
        seq = int(np.exp(rng.uniform(np.log(65), np.log(2e7 / (bs * d) + 66))))
        dtype, direction = int(rng.integers(0, 3)), int(rng.choice([_native.FSS_FWD, _native.FSS_GATED_FWD]))
        finest = _native.FssConfig(1, 16, 4 if seq <= 2048 else 8, 0)
        need = lib.fss_workspace_bytes(bs, seq, d, dtype, direction, None)
        bound = lib.fss_workspace_bytes(bs, seq, d, dtype, direction, ctypes.byref(finest))
        # (rows of an odd number of 64-channel tiles are padded to two channels per lane)
        assert need <= max(LIMIT + 4096, 2 * bound), (bs, seq, d, dtype, direction)
        assert need - 4096 <= max(LIMIT, 24 * bs * -(-d // 128) * 128 * -(-seq // 64)), (bs, seq, d, dtype, direction)


def test_a_shorter_sequence_may_need_the_larger_workspace():
    """What include/fss_scan.h tells a caller that keeps one workspace for many lengths."""
    lib = _native.lib()
    bf16, gated = _native.FSS_BF16, _native.FSS_GATED_FWD
    assert lib.fss_workspace_bytes(64, 500, 1680, bf16, gated, None) < lib.fss_workspace_bytes(64, 300, 1680, bf16, gated, None)
    assert lib.fss_workspace_bytes(8, 1000, 1007, bf16, _native.FSS_FWD, None) < lib.fss_workspace_bytes(8, 700, 1007, bf16, _native.FSS_FWD, None)
    # (one workgroup would cover these: four that share the sequence are faster, and chain)
    assert lib.fss_workspace_bytes(64, 512, 4096, bf16, gated, None) == 4096 + 24 * 64 * 4096 * 4


def test_no_plain_forward_outgrows_the_static_scratch():
    """Short odd-width forwards take tiles that need more words than the ladder's other rungs only while those stay within
    half of the static array: around the array's size the words are those of 32 steps."""
    lib = _native.lib()
    for seq in (512, 700, 1000, 1024):
        for d in (1, 63, 65, 999):
            for bs in (1, 100, 1000, 1365, 1366, 5000, 6000, 20000):
                need = lib.fss_workspace_bytes(bs, seq, d, _native.FSS_BF16, _native.FSS_FWD, None) - 4096
                widest = max(lib.fss_workspace_bytes(bs, seq, d, _native.FSS_BF16, _native.FSS_FWD,
                                                     ctypes.byref(_native.FssConfig(1, 32, w, 0))) - 4096 for w in (8, 16))
                assert need <= max(8 << 20, widest), (bs, seq, d)


def test_plans_do_not_depend_on_what_was_planned_before():
    """The plans a thread keeps are those it would compute: the same answers in another order and from another thread."""
    lib = _native.lib()
    rng = np.random.default_rng(6)
    asked = [((int(rng.integers(1, 40)), int(rng.integers(1, 3000)), int(rng.integers(1, 700))), int(rng.integers(0, 3)),
              int(rng.integers(0, 4)), int(rng.choice([4, 8, 16]))) for _ in range(300)]
    first = [choose(lib, *a) for a in asked]
    order = rng.permutation(len(asked))
    again = {int(i): choose(lib, *asked[i]) for i in list(order) + list(order[::-1])}
    assert [again[i] for i in range(len(asked))] == first
    other = []
    t = threading.Thread(target=lambda: other.extend(choose(lib, *a) for a in asked))
    t.start()
    t.join()
    assert other == first


@pytest.mark.parametrize("which", range(6), ids=["bs", "seq", "d", "dtype", "dir", "align"])
def test_kept_plans_are_told_apart_by_every_argument(which):
    """Requests that differ in one argument only, asked in turn so that they meet in the table's slots, get what a plan
    that is never kept (of a configuration of zeros) says: a lookup that left the argument out would not.  (One shape's types
    and directions never share a slot, so those two are told apart already there.)"""
    lib = _native.lib()
    rng = np.random.default_rng(8)

    def plan(request, cfg):
        out = (ctypes.c_int32 * 8)()
        rc = lib.fss_debug_chain_plan(*request, cfg, out)
        return (rc, *out) if rc == 0 else (rc,)

    zeros = ctypes.byref(_native.FssConfig())
    told_apart = 0
    for _ in range(150):
        draw = [lambda: int(rng.integers(1, 200)), lambda: int(rng.integers(65, 20000)), lambda: int(rng.integers(32, 2000)),
                lambda: int(rng.integers(0, 3)), lambda: int(rng.integers(0, 4)), lambda: int(rng.choice([2, 4, 8, 16, 32]))]
        start = [f() for f in draw]
        values = [range(3), range(4), (2, 4, 8, 16, 32)][which - 3] if which >= 3 else [draw[which]() for _ in range(12)]
        requests = [tuple(start[:which] + [int(v)] + start[which + 1:]) for v in values]
        want = [plan(r, zeros) for r in requests]
        told_apart += len(set(want)) > 1
        for i in rng.integers(0, len(requests), 4 * len(requests)):
            assert plan(requests[i], None) == want[i], requests[i]
    assert told_apart >= 50


def test_the_plans_for_all_alignments_are_kept_together():
    """fss_workspace_bytes plans a shape for 2, 4, 8 and 16 bytes: asked again, it plans nothing anew."""
    lib = _native.lib()
    rng = np.random.default_rng(7)
    for _ in range(200):
        shape = int(rng.integers(1, 64)), int(rng.integers(1, 5000)), int(rng.integers(1, 2000))
        dtype, direction = int(rng.integers(0, 3)), int(rng.integers(0, 4))
        need = lib.fss_workspace_bytes(*shape, dtype, direction, None)
        before = lib.fss_debug_plans_computed()
        assert lib.fss_workspace_bytes(*shape, dtype, direction, None) == need
        # (fp32 tensors never start at 2 bytes: that plan is refused, and refusals are not kept)
        refused = 1 if dtype == _native.FSS_F32 else 0
        assert lib.fss_debug_plans_computed() - before == refused, (shape, dtype, direction)


def test_small_and_large_forwards():
    lib = _native.lib()
    # a launch that leaves most of the device idle takes short tiles, the device's ladder begins where launches fill it
    assert choose(lib, (1, 697, 448), _native.FSS_BF16, _native.FSS_FWD)[1] == 8
    assert choose(lib, (10, 1871, 256), _native.FSS_BF16, _native.FSS_GATED_FWD) == (2, 16, 12, 1)
    assert choose(lib, (8, 2048, 1024), _native.FSS_BF16, _native.FSS_FWD) == (2, 32, 16, 1)
    # never two channels per lane where rows or tensors do not allow them
    assert choose(lib, (3, 614, 1007), _native.FSS_BF16, _native.FSS_FWD)[0] == 1
    assert choose(lib, (10, 1871, 256), _native.FSS_BF16, _native.FSS_GATED_FWD, 2)[0] == 1


def test_named_parts_of_a_tiling_keep_their_ladder():
    """A caller who names two column tiles (or steps, or waves) and leaves the rest open gets a tiling that these divide,
    at the shapes where the library's own choice has three tiles per row, twelve waves or wider lanes."""
    lib = _native.lib()
    bf16, fp16, fp32 = _native.FSS_BF16, _native.FSS_F16, _native.FSS_F32
    fwd, bwd, gfwd = _native.FSS_FWD, _native.FSS_BWD, _native.FSS_GATED_FWD
    for shape, dtype, direction, named, want in [
            ((4, 20000, 192), bf16, bwd, (0, 0, 0, 2), (2, 16, 16, 2)), ((31, 3327, 192), bf16, fwd, (0, 0, 0, 2), (2, 32, 8, 2)),
            ((34, 5677, 192), bf16, bwd, (0, 32, 0, 2), (2, 32, 8, 2)), ((64, 40, 13200), bf16, bwd, (0, 0, 0, 2), (2, 16, 4, 2)),
            ((256, 38, 3500), fp16, bwd, (0, 0, 0, 2), (2, 16, 4, 2)), ((126, 107, 13200), bf16, bwd, (8, 8, 0, 2), (8, 8, 4, 2)),
            ((3, 7752, 384), fp16, gfwd, (0, 0, 0, 2), (1, 32, 8, 2)), ((40, 751, 384), bf16, gfwd, (0, 32, 0, 2), (1, 32, 16, 2)),
            ((4000, 40, 128), fp32, gfwd, (0, 0, 0, 2), (1, 32, 2, 2)), ((7, 4958, 3711), bf16, bwd, (0, 0, 0, 1), (1, 16, 8, 1))]:
        cfg = _native.FssConfig(named[0], named[1], named[2], 0, named[3])
        out = (ctypes.c_int32 * 8)()
        assert lib.fss_debug_chain_plan(*shape, dtype, direction, 16, ctypes.byref(cfg), out) == 0, (shape, named)
        assert (out[6], out[2], out[1] * out[7], out[7]) == want, (shape, named, list(out))


# kernel, type, elements below which the estimate chooses, and what its choice may lose in the mean against the fastest
# measured tiling (what it loses, rounded up; the ladder alone loses 14, 29, 14 and 14 %)
@pytest.mark.parametrize("kernel,dtype,limit,loss", [
    ("plain", "bf16", 15 << 20, 0.035), ("gated", "bf16", 1 << 23, 0.07),
    ("plain", "fp32", 1 << 21, 0.045), ("gated", "fp32", 1 << 22, 0.06)])
def test_the_choice_is_near_the_fastest_measured_tiling(kernel, dtype, limit, loss):
    """The estimate against times of shapes that it was not fitted to (us, one launch of many)."""
    lib = _native.lib()
    code = {"bf16": _native.FSS_BF16, "fp32": _native.FSS_F32}[dtype]
    times = {}
    with open(PAIRS) as f:
        for row in csv.DictReader(f):
            if (row["kernel"], row["dtype"]) == (kernel, dtype):
                shape = tuple(int(row[k]) for k in ("bs", "seq", "d"))
                times.setdefault(shape, {})[tuple(int(row[k]) for k in ("vec", "steps", "waves", "cols"))] = float(row["us"])
    shapes = [s for s in times if s[0] * s[1] * s[2] < limit]
    assert len(shapes) >= 70
    ratios = [times[s][choose(lib, s, code, _native.FSS_FWD if kernel == "plain" else _native.FSS_GATED_FWD)] / min(times[s].values())
              for s in shapes]
    assert np.exp(np.mean(np.log(ratios))) - 1 <= loss
