"""The kernels' address arithmetic replayed on the CPU (no GPU): every global
load and store and every LDS window access of the batched MFMA kernel
(jh_mfma.hip gemm_body / mfma_px), the staged B = 1 kernel
(jh_gemv_staged.hip) and the one-shot kernels (jh_gemv.hip), for every
benchmark shape, batch and row range, must stay inside the buffer it targets.

Each model below restates one kernel's index formulas with its file:line, per
lane, wave, workgroup and step (numpy over all of them at once, at the extreme
steps), and asserts the byte range it touches against the allocation: a packed
matrix is rows x pitch bytes plus kTailPad (256) bytes of zeros
(jh_kernels.hpp:12); x is B x cols floats; y, the split-K partials, the
counters and the prepared-x slabs are sized by the planner's own formulas.
The MFMA model's plan (K split, prepared x or not) is checked against the
library's planner (jh_qmatvec_batched_plan), so the model walks the same
launches the library makes.

It was written for an unexplained hipErrorIllegalAddress seen once on the
first eager B = 32 MFMA launch of a bench run: it finds every access of the
current kernels in bounds at every benchmark configuration.
"""
import ctypes

import numpy as np
import pytest

from juno_amd import _lib

TAIL = 256  # kTailPad, jh_kernels.hpp:12
Q4_K, Q5_K, Q6_K, Q8_0, Q2_K, Q3_K = 12, 13, 14, 8, 10, 11
BLOCK = {Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), Q8_0: (32, 34), Q2_K: (256, 84), Q3_K: (256, 110)}


def pitch(t, cols):
    qk, bb = BLOCK[t]
    return cols // qk * bb


# the matrices of TinyLlama, Llama-3-8B and Phi-3-mini, and some odd ones
SHAPES = sorted({
    (Q4_K, 5632, 2048), (Q4_K, 2048, 2048), (Q4_K, 256, 2048), (Q6_K, 256, 2048), (Q6_K, 2048, 5632),
    (Q6_K, 32000, 2048),
    (Q4_K, 4096, 4096), (Q4_K, 1024, 4096), (Q6_K, 1024, 4096), (Q4_K, 14336, 4096), (Q6_K, 4096, 14336),
    (Q6_K, 128256, 4096),
    (Q8_0, 9216, 3072), (Q8_0, 3072, 3072), (Q8_0, 16384, 3072), (Q8_0, 3072, 8192), (Q8_0, 32064, 3072),
    (Q6_K, 9216, 3072), (Q6_K, 3072, 3072), (Q6_K, 16384, 3072), (Q6_K, 3072, 8192), (Q6_K, 32064, 3072),
    (Q5_K, 3072, 3072), (Q2_K, 2048, 2048), (Q3_K, 2048, 2048), (Q4_K, 333, 768), (Q6_K, 333, 768),
})


def ranges(rows):
    out = {(0, rows), (1, rows), (0, rows - 1), (rows // 3, rows - rows // 5)}
    return sorted((a, b) for a, b in out if 0 <= a < b <= rows)


def within(lo, hi, size, what):
    lo, hi = int(np.min(lo)), int(np.max(hi))
    assert lo >= 0 and hi <= size, f"{what}: bytes [{lo}, {hi}) outside [0, {size})"


# ------------------------------------------------------------------ batched MFMA kernels (jh_mfma.hip)
# kBytes, kChunks, kRowChunks and the sums of x it reads (kSums) of each format
MF = {Q4_K: (144, 9, 9, 32), Q5_K: (176, 11, 11, 32), Q6_K: (210, 14, 15, 0), Q8_0: (272, 18, 19, 0), Q2_K: (84, 6, 7, 16),
      Q3_K: (110, 8, 9, 0)}
ROWS_PER_WAVE, WAVES, ROWS_PER_WG, MIN_WG, COUNTER_SLOTS = 32, 8, 256, 256, 1024
STATIC_SCRATCH = 8 << 20
COLH = 256 + 8  # halves per column of the staged x, kXPad among them
WIN_PAD = 16
HL_MAX = 16     # kHlMaxBatch


def two_vectors_pay(t, rows, cols):
    if t not in (Q4_K, Q5_K, Q8_0):
        return False
    if t == Q8_0:
        return rows * cols >= (22e6 if rows > 2048 else 36e6)
    return rows * cols >= (26e6 if rows > 4096 else 36e6)


def plan(t, rows, cols, B):
    """plan_group for one matrix: None, or (ksb, ksplit, columns per chunk, chunks, prepared)."""
    nsb = cols // 256
    if B == 2 and not two_vectors_pay(t, rows, cols):
        return None
    tiles = -(-rows // ROWS_PER_WG)
    best = None
    for c in (64, 32) if B > 64 and t not in (Q6_K, Q3_K) else (32,):
        chunks = 1 if B <= 64 else -(-B // c)
        for ks in range(1, nsb + 1):
            ksb = -(-nsb // ks)
            kse = -(-nsb // ksb)
            if kse > 1 and (tiles * chunks > COUNTER_SLOTS or (B > 64 and 4 * kse * B * rows > STATIC_SCRATCH)):
                break
            if c == 64 and t == Q8_0 and ksb > 16:  # kLongWalk
                continue
            rounds = -(-tiles * chunks * kse // MIN_WG)
            cost = (4 * (rounds * (ksb + 5) + (kse > 1)) + (kse if kse > 1 else 0)) * (8 if c == 64 else 5)
            if best is None or cost < best[0]:
                best = (cost, ksb, kse, c, chunks)
    _, ksb, kse, c, chunks = best
    prepared = kse == 1 and B <= 32 and t not in (Q2_K, Q3_K)
    return ksb, kse, c, chunks, prepared


class Image:
    """The x of one super-block in LDS (XImage, or Slab where x is prepared): where a
    lane's values go and where operands are read, in bytes."""

    def __init__(self, hl, nt, prepared):
        self.hl, self.nt, self.prepared = hl, nt, prepared
        self.cols = 16 if hl else 32 * nt  # columns staged
        if prepared:
            self.lo = 0 if hl else 16384
            self.xs, self.x16 = (16384 if hl else 32768), 0
            self.cs = self.xs + 1024
            self.size = (self.xs // 1024 + 2) * 1024
        else:
            self.lo = 2 * (16 if hl else 32 * nt) * COLH
            self.xs = 2 * (1 if hl else 2) * 32 * nt * COLH
            self.x16 = self.xs + 2 * 32 * nt * 16
            self.cs = self.x16 + 2 * 32 * nt * 32
            self.size = self.cs + 32 * nt * 4

    def unit(self, v, off, lo):
        """Byte of the 8 values from `off` on of A row v (!hl: of its lo plane)."""
        if self.prepared:
            return (self.lo if lo else 0) + 16 * ((v << 5) | ((off >> 3) ^ v))
        return (self.lo if lo else 0) + 2 * (v * COLH + off)

    def writes(self):
        """name -> (start, length) of everything one super-block's staging writes."""
        col = np.arange(self.cols)[:, None, None]
        q, u = np.arange(16)[None, :, None], np.arange(2)[None, None, :]
        off = 16 * q + 8 * u
        out = {"hi": (self.unit(col, off, False), 16)}
        # with both limbs in one operand the lo limbs are A rows 16 .. 31
        out["lo"] = (self.unit(16 + col, off, False) if self.hl and self.prepared else self.unit(col, off, True), 16)
        rows = 32 * self.nt
        out["sums32"] = (self.xs + 2 * np.arange(rows * 16), 2)
        if not self.prepared:
            out["sums16"] = (self.x16 + 2 * np.arange(rows * 32), 2)
        out["scales"] = (self.cs + 4 * col.reshape(-1), 4)
        return out

    def reads(self):
        row, kh = np.arange(32 * self.nt)[:, None], np.arange(2)[None, :]
        off = 16 * np.arange(16)[:, None, None] + 8 * kh
        out = {"x": (self.unit(row, off, False), 16)}
        if not self.hl:
            out["xlo"] = (self.unit(row, off, True), 16)
        out["sums32"] = (self.xs + 2 * (row * 16 + 8 * kh), 16)
        if not self.prepared:
            out["sums16"] = (self.x16 + 2 * (row[..., None] * 32 + 8 * kh[..., None] + 16 * np.arange(2)), 16)
        n, i = np.arange(self.nt)[:, None, None], np.arange(2 if self.hl else 4)[None, :, None]
        out["scales"] = (self.cs + 4 * (n * 32 + 8 * i + 4 * kh[None]), 16)
        return out


def bytes_of(a):
    start, n = a
    return np.unique((np.asarray(start).reshape(-1, 1) + np.arange(n)).reshape(-1))


@pytest.mark.parametrize("hl,nt,prepared", [(True, 1, False), (False, 1, False), (False, 2, False), (True, 1, True),
                                            (False, 1, True)])
def test_x_image(hl, nt, prepared):
    """What the staging writes does not overlap and stays in the image, and what the
    operand reads touch has been written."""
    im = Image(hl, nt, prepared)
    parts = {k: bytes_of(v) for k, v in im.writes().items()}
    everything = np.concatenate(list(parts.values()))
    assert len(np.unique(everything)) == len(everything)
    within(everything, everything + 1, im.size, "x image write")
    for name, r in im.reads().items():
        assert np.all(np.asarray(r[0]) % min(r[1], 16) == 0), name
        assert np.isin(bytes_of(r), everything).all(), name


def win_chunk(j, ch, rc):
    return j + (rc - ch) * (j // ch)


def check_mfma_weights(t, rows_alloc, p, row0, nrows, tiles, sb_ranges, nt, image_bytes, lds_total, prepared):
    """RowSpan's 32-bit offsets, the weight chunk loads (JH_LOAD_W), the windows'
    writes (JH_PARK) and field reads, and the fields that run() reads in memory."""
    kbytes, ch, rc_fmt, _ = MF[t]
    rc = rc_fmt if nt == 1 else ch
    cl = (ROWS_PER_WAVE * ch + 63) // 64
    lane, k = np.arange(64), np.arange(cl)
    j = np.minimum(lane[:, None] + 64 * k[None, :], ROWS_PER_WAVE * ch - 1)           # (64, CL)
    rbase = (np.arange(tiles)[:, None] * ROWS_PER_WG + np.arange(WAVES)[None] * ROWS_PER_WAVE)[..., None, None]

    def row(rho):
        return np.minimum(rbase + rho, nrows - 1)

    first = (row0 + row(0)) * p
    base = first & ~15

    def offset(rho):
        o = (first & 15) + (row(rho) - row(0)) * p
        assert o.max() + max(b for _, b in sb_ranges) * kbytes + 16 * ch < 1 << 32
        return o

    coff, myoff = offset(j[None, None] // ch) + 16 * (j[None, None] % ch), offset((lane & 31)[None, None, :, None])
    alloc = rows_alloc * p + TAIL
    windows = 0 if prepared else (2 if nt == 1 else 1) * image_bytes  # mfma_px: an array of their own
    size = WAVES * ROWS_PER_WAVE * rc * 16 + WIN_PAD if prepared else lds_total
    wave0 = windows + np.arange(WAVES)[None, :, None, None] * (ROWS_PER_WAVE * rc * 16)
    for sb0, sb1 in sb_ranges:
        for sb in {sb0, sb1 - 1}:
            a = base + ((coff + sb * kbytes) & ~15)
            within(a, a + 16, alloc, f"mfma weights type {t} sb {sb}")
            # a row's block inside its window, read up to a dword past it (lds_read_u)
            at = wave0 + (lane & 31)[None, None, :, None] * rc * 16 + ((myoff + sb * kbytes) & 15)
            within(at, at + kbytes + 4, size, f"mfma window read type {t}")
            assert ((myoff + sb * kbytes) & 15).max() + kbytes <= 16 * ch  # the block was loaded whole
            a = base + myoff + sb * kbytes  # run(): the fields of a block, all inside it
            within(a, a + kbytes, alloc, f"mfma fp32 products type {t} sb {sb}")
    live = (lane[:, None] + 64 * k[None, :]) < ROWS_PER_WAVE * ch
    w = wave0 + 16 * win_chunk(j, ch, rc)[None, None]
    within(w[..., live], w[..., live] + 16, size, f"mfma window write type {t}")


@pytest.mark.parametrize("t,rows,cols", [s for s in SHAPES if s[2] % 256 == 0])
def test_mfma_addresses(t, rows, cols):
    L = _lib.load()
    p = pitch(t, cols)
    nsb = cols // 256
    for B in (2, 3, 8, 16, 17, 20, 31, 32, 33, 48, 64, 65, 97, 128, 130):
        for r0, r1 in ranges(rows):
            nrows = r1 - r0
            tiles = -(-nrows // ROWS_PER_WG)
            pl = plan(t, nrows, cols, B)
            # the library plans the same launch with the same layout
            kern, ks, lay = ctypes.c_int(), ctypes.c_int(), (ctypes.c_int * 13)()
            assert L.jh_qmatvec_batched_plan_shape(t, cols, r0, r1, B, ctypes.byref(kern), ctypes.byref(ks)) == 0
            assert L.jh_qmatvec_batched_layout_shape(t, cols, r0, r1, B, lay, 13) == 0
            if pl is None:
                assert kern.value == 0 and not any(lay)
                continue
            ksb, ksplit, chunk, chunks, prepared = pl
            hl = B <= HL_MAX
            nt = chunk // 32 if B > 64 else 2 if B > 32 else 1
            im = Image(hl, nt, prepared)
            kbytes, ch, rc_fmt, _ = MF[t]
            rc = rc_fmt if nt == 1 else ch
            windows = WAVES * ROWS_PER_WAVE * (rc_fmt if prepared or nt == 1 else max(rc_fmt, ch)) * 16 + WIN_PAD
            lds = (2 if nt == 1 else 1) * im.size + windows
            assert (kern.value, ks.value) == (2 if prepared else 1, ksplit), (t, rows, cols, B, r0, r1)
            assert list(lay) == [kern.value, ksplit, ksb, chunk if B > 64 else im.cols, chunks, im.lo, im.xs, im.x16, im.cs,
                                 im.size, ch, rc, lds], (t, rows, cols, B, r0, r1)
            assert lds <= 160 * 1024
            sb_ranges = [(sp * ksb, min(nsb, sp * ksb + ksb)) for sp in range(ksplit)]
            assert all(a < b for a, b in sb_ranges)
            check_mfma_weights(t, rows, p, r0, nrows, tiles, sb_ranges, nt, im.size, lds, prepared)
            plane, covered = B * nrows, 0
            for c in range(chunks):
                col0 = c * chunk if B > 64 else 0
                bc = min(32 * nt, B - col0) if B > 64 else B  # this chunk's columns
                covered += bc
                assert 1 <= bc <= im.cols
                # x (JH_LOAD_X; add_exact reads the same columns): column min(b, bc - 1) of the chunk
                last = col0 * cols + (min(im.cols - 1, bc - 1)) * cols + (nsb - 1) * 256 + 16 * 15 + 16
                within(col0 * cols * 4, last * 4, B * cols * 4, "x")
                # y and the split-K partials: b < bc, r < nrows, splits < ksplit
                last = col0 * nrows + (bc - 1) * nrows + nrows
                within(col0 * nrows * 4, last * 4, B * nrows * 4, "y")
                within(0, ((ksplit - 1) * plane + last) * 4, ksplit * plane * 4, "partials")
                if ksplit > 1:
                    within(c, (tiles - 1) * chunks + c + 1, COUNTER_SLOTS, "tile counters")
            assert covered == B
            if prepared:  # x_prep's slabs and the DMA rows
                rows_kb = im.size // 1024
                r = np.minimum(np.arange(WAVES)[:, None] + WAVES * np.arange(-(-rows_kb // WAVES)), rows_kb - 1)
                src = (nsb - 1) * im.size + 16 * 63 + 1024 * r
                within(src, src + 16, nsb * im.size, "prepared x slab DMA source")
                within(1024 * r, 1024 * r + 16 * 64, im.size, "prepared x slab DMA target")
                assert set(r.reshape(-1)) == set(range(rows_kb))


# ------------------------------------------------------------------ staged B = 1 kernel (jh_gemv_staged.hip)
# Fmt (jh_gemv_staged.hip:256-259): QK, BB, LPB, TBMAX, CH (16-byte chunks per row tile)
SF = {Q4_K: (256, 144, 4, 16, 145), Q5_K: (256, 176, 4, 16, 177), Q6_K: (256, 210, 4, 16, 212), Q8_0: (32, 34, 1, 64, 138)}


def staged_layouts(t, cols):
    qk, bb, lpb, tbmax, ch = SF[t]
    nb = cols // qk
    gw = 1 if nb <= tbmax else 2 if nb <= 2 * tbmax else 4  # launch_staged_t
    tb = (nb + gw - 1) // gw
    return nb, gw, tb


@pytest.mark.parametrize("t,rows,cols", [s for s in SHAPES if s[0] in SF])
def test_staged_addresses(t, rows, cols):
    qk, bb, lpb, tbmax, ch = SF[t]
    p = pitch(t, cols)
    nb, gw, tb = staged_layouts(t, cols)
    if nb > 4 * tbmax:
        pytest.skip("wider than the staged kernel takes (staged_supported)")
    K = (ch + 63) // 64                                     # loads per lane per row (:639)
    lane = np.arange(64)
    for r0, r1 in ranges(rows):
        nrows = r1 - r0
        for tile in range(gw):
            b0 = tile * tb
            ntile = min(tb, nb - b0)
            tile_bytes = ntile * bb
            nch = (15 + tile_bytes + 15) >> 4               # :672
            ld = 16 * np.minimum(lane[:, None] + 64 * np.arange(K)[None, :], nch - 1)
            assert nch <= ch, (t, cols, tile)  # every loaded chunk is parked (park: chunks < CH, :767-772)
            for vr in {0, nrows - 1}:                        # issue(): rows clamped to nrows - 1 (:743-752)
                off = (r0 + vr) * p + b0 * bb
                base = off & ~15
                within(base + ld, base + ld + 16, rows * p + TAIL, f"staged weights type {t} tile {tile}")
            # block_dot reads a block's fields from the parked row at lane_blk + cstart (cstart =
            # the row's misalignment mod 16); the last byte read past the block's start:
            # Q4_K / Q5_K the block, Q6_K dwords 0..53 of the dword-aligned start (lds_word reads
            # w[k + 1], :78-80; d at word 52), Q8_0 dwords up to 9 (:540-545)
            act_blk = (lane // lpb) < ntile
            lane_blk = np.where(act_blk, lane // lpb, 0) * bb
            field_end = {Q4_K: 144, Q5_K: 176, Q6_K: 216, Q8_0: 40}[t]
            cstart = 15 if t in (Q6_K, Q8_0) else 0  # K-quant rows are 16-byte aligned (pitch 144 / 176 x n)
            within(lane_blk, lane_blk + cstart + field_end, 16 * ch, f"staged block fields type {t}")
        # x (x_load4, :104-106): c clamped to cols - 4, so [0, cols) floats
        within(0, cols * 4, cols * 4, "staged x")


# ------------------------------------------------------------------ one-shot kernels (jh_gemv.hip)
@pytest.mark.parametrize("t,rows,cols", SHAPES)
def test_one_shot_addresses(t, rows, cols):
    """gemv_q4k_body and its siblings: row pointers clamped to nrows - 1
    (jh_gemv.hip:56-57), blocks b < nb, each field read inside its block except
    the dword realignment of 2-byte-aligned Q6_K / Q8_0 / Q3_K fields, which reads
    at most 6 bytes past a block (covered by the tail padding)."""
    qk, bb = BLOCK[t]
    p = pitch(t, cols)
    nb = cols // qk
    over = {Q4_K: 0, Q5_K: 0, Q6_K: 6, Q8_0: 6, Q2_K: 0, Q3_K: 6}[t]
    for r0, r1 in ranges(rows):
        last = (r1 - 1) * p + (nb - 1) * bb
        within(r0 * p, last + bb + over, rows * p + TAIL, f"one-shot type {t}")
