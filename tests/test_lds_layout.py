"""CPU model of the grouped GEMM's LDS layouts (parallel_amd/csrc/grouped_gemm.hip).

The kernel's DMA (buffer_load_dwordx4 ... lds) fills each 1 KiB block lane by
lane, so a lane fetches whichever global 16-byte chunk belongs at its slot;
fragment reads then locate each element with a per-lane offset.  This model
evaluates the swizzles and both sides' index expressions as the kernel's source
has them and checks (1) that the reader finds every element where the writer
put it and (2) that every read pass touches distinct banks of the 64-bank (256
B/clk) gfx950 LDS: 16 lanes per ds_read_b128 pass, 32 lanes per
ds_read_b64_tr_b16 pass.  A swizzle designed for 32 banks fails (2), which is
what the SQ_LDS_BANK_CONFLICT counter showed on the GPU before the change.
"""

import re
from pathlib import Path

import pytest

SOURCE = (Path(__file__).resolve().parents[1] / "parallel_amd" / "csrc" / "grouped_gemm.hip").read_text()


def _expression(pattern):
    """The one C expression that ``pattern`` captures in the kernel's source, as a Python function of its
    variables (integers, so / is //; swizzle templates take BK by name)."""
    found = {" ".join(f.split()) for f in re.findall(pattern, SOURCE, re.S)}
    assert len(found) == 1, f"{pattern}: {found}"
    text = re.sub(r"kc_swizzle<BK>\((\w+)\)", r"kc_swizzle(\1, BK)", found.pop()).replace("/", "//")
    text = re.sub(r"\((\w+) \? (\w+) : (\w+)\)", r"(\2 if \1 else \3)", text)
    text = re.sub(r"^(.*?) \? (.*?) : (.*)$", r"(\2) if (\1) else (\3)", text)
    code = compile(text.strip(), pattern, "eval")
    return lambda **names: eval(code, {"kc_swizzle": kc_swizzle, "mc_swizzle": mc_swizzle,  # noqa: S307
                                       "stg_swizzle": stg_swizzle, **names})


_kc, _mc, _stg = (_expression(rf"constexpr int {name}\(int \w+\) {{\s*return (.*?);")
                  for name in ("kc_swizzle", "mc_swizzle", "stg_swizzle"))


def kc_swizzle(r, BK=32):
    return _kc(r=r, BK=BK)


def mc_swizzle(kk):
    return _mc(kk=kk)


def stg_swizzle(r):
    return _stg(r=r)


# DMA: the K-contiguous row and k that a lane's 16 bytes belong to, the M/N-contiguous k-row and column.
DMA_KC_ROW = _expression(r"const int r = (li \* RPI \+ [^;]*);")
DMA_KC_K = _expression(r"dma_k\[j\] = (\(\(lane % CPR\)[^;]*);")
DMA_MC_KROW = _expression(r"dma_k\[j\] = (li \* \(64 / cpk\)[^;]*);")
DMA_MC_COL = _expression(r"const int col = \(is_a \? dt\.m0 : dt\.n0\) \+ (\(\(lane % [^;]*);")
# Fragment reads.
READ_KC = _expression(r"const int lane_off = ([^;]*);")
READ_KC_B = _expression(r"b_kc\[ks\] = B_OFF \+ ([^;]*);")
READ_KC_T = _expression(r"base \+ b_kc\[ks\] \+ ([^)]*)\);")
TR_KROW = _expression(r"const int tr_krow = ([^;]*);")
TR_COL = _expression(r"const int tr_col = ([^;]*);")
HALF8 = _expression(r"const int half8 = ([^;]*);")
READ_MC = _expression(r"b_mc\[t\] = B_OFF \+ ([^;]*);")
READ_MC_KS = _expression(r"tr_read\(base \+ b_mc\[t\] \+ ([^,]*),")
READ_MC_HI = _expression(r"\(lds_i16x4_t\*\)\(at \+ ([^)]*)\)\);")
# The row and first column of a lane's run e of four results in a 32 x 64 pass, by the MFMA (16x16x32, 32x32x16).
RUN_ROW = [_expression(r"Run\{make_float4\(c\[0\][^)]*\), (16[^,]*),"),
           _expression(r"Run\{make_float4\(c\[4 [^)]*\), ([^,]*),")]
RUN_COL = [_expression(r"Run\{make_float4\(c\[0\][^)]*\), 16[^,]*, ([^}]*)\}"),
           _expression(r"Run\{make_float4\(c\[4 [^)]*\), [^,]*, ([^}]*)\}")]
# Epilogue staging.
STG_AT = _expression(r"auto stg_at = .*?return ([^;]*);")
STG_ROW = _expression(r"auto stg_row = .*?\(slot \+ ([^;]*)\);")
STG_SWAP = _expression(r"return M32 && (\(r & 16\)) \? make_uint4\(v\.z, v\.w, v\.x, v\.y\) : v;")
STG_C8 = _expression(r"uint4 v = stg_row\(r, ([^;]*)\);")
STG_GATE = _expression(r"const uint4 gv = stg_row\(r, ([^,]*)\), uv")
STG_UP = _expression(r", uv = stg_row\(r, ([^;]*)\);")


def bank_conflicts(addrs, lanes_per_pass, width):
    n = 0
    for p in range(0, len(addrs), lanes_per_pass):
        banks = [((a // 4) + b) % 64 for a in addrs[p:p + lanes_per_pass] for b in range(width // 4)]
        n += len(banks) - len(set(banks))
    return n


def check_kc(R, swz, bk=32):
    """A K-contiguous [R rows][bk] tile, with the kernel's swizzle or another."""
    c = dict(BK=bk, RB=2 * bk, CPR=bk // 8, RPI=64 * 8 // bk, WTN=R, wn=0, kc_swizzle=lambda r, BK: swz(r))
    where = {}
    for li in range(R * c["RB"] // 1024):
        for lane in range(64):
            r = DMA_KC_ROW(li=li, lane=lane, **c)
            where[(r, DMA_KC_K(lane=lane, r=r, **c) // 8)] = li * 1024 + lane * 16
    conflicts = 0
    for t in range(R // 16):  # a fragment: 16 rows x 32 k
        for ks in range(bk // 32):
            addrs = []
            for lane in range(64):
                i16, q16 = lane & 15, lane >> 4
                lane_off = READ_KC(i16=i16, q16=q16, ks=ks, **c)
                off = READ_KC_B(lane_off=lane_off, **c) + READ_KC_T(t=t, **c)
                assert where[(16 * t + i16, 4 * ks + q16)] == off
                addrs.append(off)
            conflicts += bank_conflicts(addrs, 16, 16)
    return conflicts


def check_mc(R, WT, swz, bk=32, M32=0):
    """An M/N-contiguous [bk k-rows][R columns] tile, a wave's columns being WT wide."""
    c = dict(BM=R, BN=R, WTN=WT, is_a=False, cpk=R // 8, mc_swizzle=swz)
    where = {}
    for li in range(R * bk * 2 // 1024):
        for lane in range(64):
            kk = DMA_MC_KROW(li=li, lane=lane, **c)
            col = DMA_MC_COL(lane=lane, dma_k=[kk], j2=0, **c)
            where[(kk, col // 8)] = li * 1024 + lane * 16
    conflicts = 0
    FR, FK = (32, 16) if M32 else (16, 32)
    c.update(FR=FR, FK=FK, M32=M32)
    for wn in range(R // WT):
        for t in range(WT // FR):  # a fragment: FR columns x FK k, two transpose reads
            for ks in range(bk // FK):
                for h in range(2):
                    addrs = []
                    for lane in range(64):
                        i16, q16 = lane & 15, lane >> 4
                        krow, col = TR_KROW(i16=i16, q16=q16, M32=M32), TR_COL(i16=i16, q16=q16, M32=M32)
                        off = (READ_MC(tr_krow=krow, tr_col=col, half8=HALF8(i16=i16), wn=wn, t=t, **c)
                               + READ_MC_KS(ks=ks, **c) + h * READ_MC_HI(row_bytes=R * 2))
                        # The transpose hands lane l (column l % FR) the k's 8 (l / FR) + 4 h ..: the lanes that
                        # read them are the 16 of l's quarter.
                        k0, col0 = FK * ks + 8 * (lane // FR) + 4 * h, wn * WT + FR * t + (lane % FR) // 16 * 16
                        kr, gcol = k0 + (i16 >> 2), col0 + 4 * (i16 & 3)
                        assert where[(kr, gcol >> 3)] + (gcol & 7) * 2 == off
                        addrs.append(off)
                    conflicts += bank_conflicts(addrs, 32, 8)
    return conflicts


@pytest.mark.parametrize("M32", [0, 1])
def test_epilogue_staging_is_consistent_and_conflict_free(M32):
    """A wave's 32 x 64 bf16 pass: 8-byte writes of runs of four columns, then row reads and (16x16x32 only)
    the SwiGLU gate/up reads of whole 16-byte chunks, with the halves of rows 16 .. 31 in exchange for 32x32x16."""
    where = {}
    for e in range(8):
        addrs = []
        for lane in range(64):
            names = dict(i16=lane & 15, q16=lane >> 4, l32=lane & 31, khalf=lane >> 5, e=e)
            row, col = RUN_ROW[M32](**names), RUN_COL[M32](**names)
            addrs.append(STG_AT(row=row, col=col, M32=M32))
            where[(row, col)] = addrs[-1]
        assert bank_conflicts(addrs, 32, 8) == 0
    assert len(where) == len(set(where.values())) == 32 * 16

    def reads(rows, chunks):
        addrs = [STG_ROW(r=r, chunk=c) for r, c in zip(rows, chunks)]
        for r, c, a in zip(rows, chunks, addrs):
            swap = 8 if M32 and STG_SWAP(r=r) else 0
            assert where[(r, 8 * c)] == a + swap and where[(r, 8 * c + 4)] == a + 8 - swap
        assert bank_conflicts(addrs, 16, 16) == 0

    lanes = range(64)
    for n in range(4):
        reads([8 * n + (lane >> 3) for lane in lanes], [STG_C8(c8=lane & 7) for lane in lanes])
    for n in range(0 if M32 else 2):
        rows = [16 * n + (lane >> 2) for lane in lanes]
        reads(rows, [STG_GATE(c4=lane & 3) for lane in lanes])
        reads(rows, [STG_UP(c4=lane & 3) for lane in lanes])


@pytest.mark.parametrize("R", [128, 256])
def test_k_contiguous_layout_is_consistent_and_conflict_free(R):
    assert check_kc(R, kc_swizzle) == 0


@pytest.mark.parametrize("M32", [0, 1])
@pytest.mark.parametrize("R,WT", [(128, 64), (256, 64), (256, 128)])
def test_transpose_read_layout_is_consistent_and_conflict_free(R, WT, M32):
    assert check_mc(R, WT, mc_swizzle, M32=M32) == 0


@pytest.mark.parametrize("R", [64, 128, 256])
def test_64_deep_layouts_are_consistent_and_conflict_free(R):
    assert check_kc(R, lambda r: kc_swizzle(r, 64), bk=64) == 0
    if R >= 128:
        assert check_mc(R, 64, mc_swizzle, bk=64) == 0
        assert check_mc(R, 64, mc_swizzle, bk=64, M32=1) == 0


def test_model_flags_32_bank_swizzles():
    assert check_kc(256, lambda r: (r >> 1) & 3) > 0
    assert check_mc(256, 64, lambda kk: 2 * (kk & 3)) > 0
