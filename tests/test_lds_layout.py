"""CPU model of the grouped GEMM's LDS layouts (parallel_amd/csrc/grouped_gemm.hip).

The kernel's DMA (buffer_load_dwordx4 ... lds) fills each 1 KiB block lane by
lane, so a lane fetches whichever global 16-byte chunk belongs at its slot;
fragment reads then locate each element with a per-lane offset.  This model
restates both sides' index formulas and checks (1) that the reader finds
every element where the writer put it and (2) that every read pass touches
distinct banks of the 64-bank (256 B/clk) gfx950 LDS: 16 lanes per
ds_read_b128 pass, 32 lanes per ds_read_b64_tr_b16 pass.  A swizzle designed
for 32 banks fails (2), which is what the SQ_LDS_BANK_CONFLICT counter showed
on the GPU before the change.
"""

import pytest


def kc_swizzle(r):  # K-contiguous: row bits 2-3
    return (r >> 2) & 3


def mc_swizzle(kk):  # M/N-contiguous: k-row & 3 selects the 64-byte bank quarter, bit 3 the half of it
    return 4 * (kk & 3) | 2 * ((kk >> 3) & 1)


def bank_conflicts(addrs, lanes_per_pass, width):
    n = 0
    for p in range(0, len(addrs), lanes_per_pass):
        banks = [((a // 4) + b) % 64 for a in addrs[p:p + lanes_per_pass] for b in range(width // 4)]
        n += len(banks) - len(set(banks))
    return n


def check_kc(R, swz, bk=32):
    cpr = bk // 8  # chunks of 16 B per row of a k-tile
    rb = 2 * bk
    where = {}
    for li in range(R * rb // 1024):
        for lane in range(64):
            r = li * (64 // cpr) + lane // cpr
            where[(r, (lane % cpr) ^ swz(r))] = li * 1024 + lane * 16
    conflicts = 0
    for row0 in range(0, R, 16):  # a fragment: 16 rows x 32 k
        for ks in range(bk // 32):
            addrs = []
            for lane in range(64):
                i16, q = lane & 15, lane >> 4
                off = row0 * rb + i16 * rb + (((4 * ks + q) ^ swz(i16)) << 4)
                assert where[(row0 + i16, 4 * ks + q)] == off
                addrs.append(off)
            conflicts += bank_conflicts(addrs, 16, 16)
    return conflicts


def check_mc(R, WT, swz, bk=32):
    cpk = R // 8
    where = {}
    for li in range(R * bk * 2 // 1024):
        for lane in range(64):
            kk = li * (64 // cpk) + lane // cpk
            where[(kk, (lane % cpk) ^ swz(kk))] = li * 1024 + lane * 16
    conflicts = 0
    for wcb in range(0, R, WT):
        for t in range(WT // 16):  # a fragment: 16 columns x 32 k, two transpose reads
            for ks in range(bk // 32):
                for h in range(2):
                    addrs = []
                    for lane in range(64):
                        q, i = lane >> 4, lane & 15
                        krow = 8 * q + (i >> 2)
                        col = 4 * (i & 3)
                        off = (krow * R * 2 + ((((wcb + 16 * t + col) >> 3) ^ swz(krow)) << 4)
                               + ((i & 1) << 3) + 32 * ks * R * 2 + h * 4 * R * 2)
                        kr, gcol = 32 * ks + krow + 4 * h, wcb + 16 * t + col
                        assert where[(kr, gcol >> 3)] + (gcol & 7) * 2 == off
                        addrs.append(off)
                    conflicts += bank_conflicts(addrs, 32, 8)
    return conflicts


def test_epilogue_staging_is_conflict_free():
    """A wave's 32 x 64 bf16 pass: 8-byte writes (row 16 hh + i16, chunk 2 tt + q16 / 2, half q16 & 1),
    then row reads and the SwiGLU gate/up reads of whole chunks."""
    def at(r, chunk):
        return r * 128 + ((chunk ^ ((((r >> 1) & 1) << 2) | ((r >> 2) & 3))) << 4)

    for hh in range(2):
        for tt in range(4):
            writes = [at(16 * hh + (l & 15), 2 * tt + (l >> 5)) + ((l >> 4 & 1) << 3) for l in range(64)]
            assert bank_conflicts(writes, 32, 8) == 0
    for n in range(4):
        assert bank_conflicts([at(8 * n + (l >> 3), l & 7) for l in range(64)], 16, 16) == 0
    for n in range(2):
        for half in (0, 4):
            assert bank_conflicts([at(16 * n + (l >> 2), (l & 3) + half) for l in range(64)], 16, 16) == 0


@pytest.mark.parametrize("R", [128, 256])
def test_k_contiguous_layout_is_consistent_and_conflict_free(R):
    assert check_kc(R, kc_swizzle) == 0


@pytest.mark.parametrize("R,WT", [(128, 64), (256, 64), (256, 128)])
def test_transpose_read_layout_is_consistent_and_conflict_free(R, WT):
    assert check_mc(R, WT, mc_swizzle) == 0


@pytest.mark.parametrize("R", [64, 128, 256])
def test_64_deep_layouts_are_consistent_and_conflict_free(R):
    assert check_kc(R, lambda r: (r >> 1) & 7, bk=64) == 0
    if R >= 128:
        assert check_mc(R, 64, mc_swizzle, bk=64) == 0


def test_model_flags_32_bank_swizzles():
    assert check_kc(256, lambda r: (r >> 1) & 3) > 0
    assert check_mc(256, 64, lambda kk: 2 * (kk & 3)) > 0
