"""Host-side checks of which tilings large launches take: on both sides of each line that a rule draws."""
import csv
import ctypes
from pathlib import Path

import numpy as np
import pytest

from fast_sequential_scan_amd import _native

BF16, F32, FP16 = _native.FSS_BF16, _native.FSS_F32, _native.FSS_F16
FWD, BWD, GATED_FWD = _native.FSS_FWD, _native.FSS_BWD, _native.FSS_GATED_FWD


def choose(shape, dtype, direction, align=16):
    cfg = _native.FssConfig()
    assert _native.lib().fss_choose_config(*shape, dtype, direction, align, ctypes.byref(cfg)) == 0
    return cfg.vec, cfg.steps, cfg.waves, cfg.cols


# backwards of rows that are no whole number of 64-byte sectors: 12 waves, and each reason for 16
@pytest.mark.parametrize("shape,waves", [
    ((27, 8422, 210), 12), ((26, 3001, 526), 12), ((1, 14448, 2346), 12),
    ((26, 5000, 210), 16),                                          # below 2^25 elements
    ((27, 8422, 224), 16), ((27, 8422, 256), 16),                   # whole sectors
    ((48, 17050, 82), 16), ((64, 8422, 126), 16),                   # one column tile per row: no seam
    ((43, 235, 3380), 16), ((60, 407, 1424), 16),                   # 192-step chunks pad an eighth further
    ((10, 1190, 3804), 12), ((130, 1745, 342), 12),                 # a twentieth and a fourteenth
    ((54, 608, 2168), 16), ((20, 640, 3828), 16), ((40, 641, 4008), 12),  # four chunks for three, the last nearly empty
    ((90, 265, 1458), 12), ((190, 256, 1458), 16), ((24, 956, 2034), 12),  # few chunks
    ((1362, 124, 692), 12), ((445, 97, 1938), 12), ((582, 84, 2186), 8), ((256, 96, 3158), 8), ((420, 51, 3588), 6),  # one, of as many
    ((330, 64, 3588), 6), ((700, 48, 1676), 4),                            # waves as the steps need
    ((340, 457, 222), 12), ((340, 448, 222), 16), ((114, 512, 700), 12), ((114, 513, 700), 12),  # the third chunk a third full
    ((3249, 269, 112), 12), ((470, 800, 112), 16),                         # one column tile: three chunks for four
    ((4, 25461, 382), 12), ((1, 51198, 794), 12), ((14, 54771, 174), 12),  # a long chain
    ((14, 51817, 144), 16), ((14, 51817, 146), 12)])
def test_backward_of_sector_sharing_rows(shape, waves):
    for dtype in (BF16, FP16):
        assert choose(shape, dtype, BWD) == (2, 16, waves, 1), shape


# backwards of odd width: 16 waves from 2^25 elements on, where their chunks do not pad the sequence much further and rows are not narrow
@pytest.mark.parametrize("shape,waves", [
    ((75, 11521, 71), 8), ((171, 8554, 85), 8), ((171, 8554, 89), 16), ((179, 8888, 47), 8),
    ((7, 4958, 3767), 16), ((4, 8354, 1531), 16), ((20, 1072, 1817), 16), ((48, 185, 3847), 16),
    ((31, 607, 1041), 8),                                           # below 2^25 elements
    ((57, 261, 2529), 8), ((28, 525, 2681), 8), ((40, 870, 3567), 16),  # 512, 768 and 1024 for 384, 640 and 896
    ((512, 66, 3475), 8), ((190, 128, 2633), 8), ((113, 137, 3563), 16), ((48, 12642, 61), 8)])  # 8 waves cover it; narrow
def test_backward_of_odd_width(shape, waves):
    for dtype in (BF16, FP16):
        assert choose(shape, dtype, BWD) == (1, 16, waves, 1), shape
    # (tensors of even width that start at an odd element are the same case)
    assert choose((shape[0], shape[1], shape[2] + 1), BF16, BWD, 2) == (1, 16, waves, 1)


def test_backward_of_rows_of_one_whole_tile():
    for shape, waves in [((48, 12642, 64), 16), ((2721, 214, 64), 16), ((1825, 426, 64), 16), ((3121, 266, 64), 8)]:  # 512 for 384
        assert choose(shape, BF16, BWD) == (1, 16, waves, 1), shape


def test_backward_of_odd_width_and_few_steps():
    for shape in [(577, 60, 3709), (880, 51, 1161), (600, 64, 1161)]:
        assert choose(shape, BF16, BWD) == (1, 8, 8, 1), shape


# forwards of odd width and up to 1024 steps: 128-step chunks where they pad a fifth less than 512-step ones
@pytest.mark.parametrize("shape,steps", [
    ((29, 574, 1319), 16), ((23, 749, 1927), 16), ((24, 384, 1735), 16), ((33, 561, 2107), 16),
    ((36, 393, 1921), 32), ((62, 1000, 343), 32), ((13, 872, 1465), 32),  # 512 for 512, 1024 for 1024 and 896
    ((35, 169, 2995), 32), ((53, 188, 2485), 32), ((61, 254, 3011), 32),  # one chunk of 256 steps
    ((208, 59, 97), 16), ((35, 38, 2715), 16), ((2675, 20, 113), 16), ((150, 64, 1735), 16), ((180, 65, 1735), 32),  # up to 64 steps
    ((24, 1300, 1735), 32),                                               # more than 1024 steps
    ((85, 588, 1999), 32)])                                               # words beyond half the static array
def test_forward_of_odd_width(shape, steps):
    for dtype in (BF16, FP16):
        assert choose(shape, dtype, FWD)[:2] == (1, steps), shape
    assert choose((shape[0], shape[1], shape[2] + 1), BF16, FWD, 2)[:2] == (1, steps)


# gated forwards of fp32 from 4 Mi elements on: 12 waves, or 8 where 12 pad the sequence by more than a tenth; the ladder's where one
# of its tiles covers the sequence and the last wave has fewer than 16 of 32 steps, in rows of whole sectors
@pytest.mark.parametrize("shape,want", [
    ((10, 24028, 128), (1, 16, 12, 1)), ((11, 1623, 1152), (1, 16, 12, 1)), ((9, 7795, 67), (1, 16, 12, 1)),
    ((34, 214, 664), (1, 16, 8, 1)), ((229, 444, 256), (1, 16, 8, 1)), ((60, 80, 1024), (1, 16, 8, 1)), ((41, 430, 3648), (1, 32, 16, 1)),
    ((42, 196, 2368), (1, 32, 8, 1)), ((60, 78, 1024), (1, 32, 4, 1)), ((142, 386, 1088), (1, 32, 16, 1)), ((92, 96, 3328), (1, 32, 4, 1)),
    ((41, 417, 3646), (1, 16, 8, 1)), ((45, 590, 3264), (1, 16, 8, 1)),  # rows that share sectors; more than 512 steps
    ((30, 322, 3264), (1, 16, 12, 1)),                              # 384 steps either way
    ((59, 47, 3904), (1, 16, 4, 1)), ((24, 55, 3756), (1, 16, 4, 1)), ((43, 32, 3345), (1, 16, 2, 1)),
    ((8, 4096, 1024), (1, 32, 16, 1))])                             # whole rounds of the largest tile
def test_gated_forward_in_single_precision(shape, want):
    assert choose(shape, F32, GATED_FWD) == want


# rows of three 64-channel tiles: one channel per lane in large launches
def test_rows_of_three_column_tiles():
    for dtype in (BF16, FP16):
        for shape in [(4, 57534, 192), (7, 30000, 192), (30, 13002, 192), (11, 56047, 192), (12, 14564, 192)]:
            assert choose(shape, dtype, FWD) == (1, 32, 8, 1), shape
        for shape in [(591, 268, 192), (878, 284, 192), (350, 512, 192)]:  # one chunk of 16 waves
            assert choose(shape, dtype, FWD)[:2] == (2, 32), shape
        # (words beyond the static array of the forward that allocates nothing, which takes these shapes otherwise)
        for shape in [(2, 480000, 192), (1000, 1000, 192)]:
            assert choose(shape, dtype, FWD)[0] == 2
            assert _native.lib().fss_workspace_bytes(*shape, dtype, FWD, None) <= 16 << 20, shape
        for shape in [(4, 20000, 192), (30, 2000, 192), (8, 40000, 192)]:
            assert choose(shape, dtype, BWD) == (1, 16, 16, 1), shape
        assert choose((20, 2000, 192), dtype, BWD)[0] == 2  # below 2^23 elements
        for d in (128, 256, 320):
            assert choose((8, 20000, d), dtype, FWD)[0] == 2 and choose((8, 20000, d), dtype, BWD)[0] == 2
    # fp32 has one channel per lane at these widths anyhow
    assert choose((4, 57534, 192), F32, FWD)[0] == 1


# gated forwards of just the size from which launches count as filling the device: the ladder's tile where it has one round
@pytest.mark.parametrize("shape,dtype,want", [
    ((16, 2048, 256), BF16, (2, 16, 16, 1)), ((32, 256, 1024), BF16, (2, 16, 16, 1)), ((8, 1024, 1024), FP16, (2, 16, 16, 1)),
    ((8, 4096, 256), BF16, (1, 32, 16, 1)), ((1, 32768, 256), BF16, (1, 32, 16, 1)), ((16, 8192, 64), BF16, (1, 32, 16, 1)),
    ((64, 128, 1024), BF16, (2, 16, 8, 1)), ((64, 2048, 64), BF16, (1, 16, 12, 1)),  # no one round of a 16-wave tile
    ((9, 1695, 1792), BF16, (2, 16, 8, 1)),                                         # above that size
    ((8, 2048, 256), F32, (1, 16, 16, 1)), ((1, 16384, 256), F32, (1, 16, 16, 1)), ((256, 64, 256), F32, (1, 16, 4, 1)),
    ((8, 2049, 256), F32, (1, 16, 12, 1))])
def test_gated_forward_of_one_round(shape, dtype, want):
    assert choose(shape, dtype, GATED_FWD) == want


# gated forwards in 16 bits of rows that share sectors and one chunk: the largest tile in many rounds
@pytest.mark.parametrize("shape,want", [
    ((129, 410, 3944), (2, 32, 16, 1)), ((83, 512, 3450), (2, 32, 16, 1)), ((256, 385, 1182), (2, 32, 16, 1)),
    ((129, 410, 3936), (2, 16, 4, 1)), ((2429, 416, 86), (2, 16, 4, 1)),    # whole sectors; narrow rows
    ((116, 455, 1948), (2, 16, 8, 1)),                                      # 7.25 rounds
    ((142, 384, 3450), (2, 16, 8, 1)), ((142, 513, 3450), (2, 16, 4, 1))])  # padded by a third; two chunks
def test_gated_forward_of_one_chunk_that_shares_sectors(shape, want):
    for dtype in (BF16, FP16):
        assert choose(shape, dtype, GATED_FWD) == want


# gated forwards in fp32 that the largest tile does not fill the device with: not 12 waves where they begin a second round
@pytest.mark.parametrize("shape,want", [
    ((7, 5420, 175), (1, 16, 16, 1)), ((2, 1306, 2560), (1, 16, 16, 1)), ((1, 1654, 3712), (1, 16, 8, 1)), ((1, 17185, 384), (1, 16, 8, 1)),
    ((1, 14009, 448), (1, 16, 12, 1)),                              # 511 tiles of 12 waves, 512 have a place
    ((1, 9031, 896), (1, 16, 12, 1)),                               # a second round that is no longer short
    ((29, 1522, 142), (1, 16, 12, 1)), ((65, 366, 1217), (1, 16, 12, 1))])  # the largest tile fills the device
def test_gated_forward_in_single_precision_without_a_short_second_round(shape, want):
    assert choose(shape, F32, GATED_FWD) == want


# gated forwards in fp32 of wide rows that share sectors: the largest tile in large launches that it does not pad much
@pytest.mark.parametrize("shape,want", [
    ((44, 1451, 1809), (1, 32, 16, 1)), ((6, 12955, 2369), (1, 32, 16, 1)), ((98, 1664, 1286), (1, 32, 16, 1)),
    ((35, 1451, 1630), (1, 16, 12, 1)),                             # below 80 Mi elements
    ((60, 1451, 1270), (1, 16, 12, 1)),                             # narrower
    ((44, 1451, 1808), (1, 16, 12, 1)),                             # whole sectors
    ((44, 1200, 1809), (1, 16, 12, 1)), ((77, 449, 3374), (1, 16, 8, 1))])  # padded by more than a quarter; one chunk
def test_gated_forward_in_single_precision_of_wide_rows_that_share_sectors(shape, want):
    assert choose(shape, F32, GATED_FWD) == want


PAIRS = Path(__file__).resolve().parent.parent / "profiles" / "large_tilings_pairs.csv"


# what the choice may lose in the mean against the fastest measured tiling (what it loses, rounded up; the ladder alone 5, 8 and 9 %)
@pytest.mark.parametrize("kernel,dtype,loss", [("backward", "bf16", 0.01), ("gated", "bf16", 0.025), ("gated", "fp32", 0.035)])
def test_the_choice_is_near_the_fastest_measured_tiling(kernel, dtype, loss):
    times = {}
    with open(PAIRS) as f:
        for row in csv.DictReader(f):
            if (row["kernel"], row["dtype"]) == (kernel, dtype):
                shape = tuple(int(row[k]) for k in ("bs", "seq", "d"))
                times.setdefault(shape, {})[tuple(int(row[k]) for k in ("vec", "steps", "waves", "cols"))] = float(row["us"])
    direction = BWD if kernel == "backward" else GATED_FWD
    chosen = {s: choose(s, BF16 if dtype == "bf16" else F32, direction) for s in times}
    ratios = [times[s][c] / min(times[s].values()) for s, c in chosen.items() if c in times[s]]
    assert len(ratios) >= 300  # (some short sequences take a tiling that was not among the named ones)
    assert np.exp(np.mean(np.log(ratios))) - 1 <= loss
