"""The tile kernel's index arithmetic (paia-project_amd/csrc/gemv_tile.h) replayed on the CPU: every tile has one unit and
every stage one wave, the XCD order is a permutation, the metadata items divide exactly and stay in their LDS words, and the
swizzled LDS layouts bring each lane the columns its MFMA step takes, without a bank conflict among 8 rows. Also its INT4
decode: nibbles as e4m3 bytes, their pairs against the re-paired activations, and the powers of two on the way."""
import re
from pathlib import Path

import numpy as np
import pytest

from test_batch_emulation import step_col


@pytest.mark.parametrize("tiles,blocks,units", [(1, 1, 1), (257, 129, 1), (632, 211, 1), (2063, 768, 1), (1792, 224, 2),
                                                (7, 1, 2), (6250, 1563, 1)])
def test_tiles_and_blocks(tiles, blocks, units):
    tq, tr = divmod(tiles, blocks * units)
    at = lambda u: u * tq + min(u, tr)
    assert at(0) == 0 and at(blocks * units) == tiles
    assert {at(u + 1) - at(u) for u in range(blocks * units)} <= {tq, tq + 1}
    per, rem = divmod(blocks, 8)
    order = [(x * (per + 1) if x < rem else rem * (per + 1) + (x - rem) * per) + b // 8
             for b in range(blocks) for x in [b % 8]]
    assert sorted(order) == list(range(blocks))


def test_most_rows():
    """At the most rows the launch takes (short rows: rounds of three blocks of 256 threads per CU, at most four tiles each),
    fewer than 2^32 threads and FP8 scales within a 32-bit buffer size."""
    src = (Path(__file__).resolve().parent.parent / "paia-project_amd/csrc/gemv_tile.hip").read_text()
    most = eval(re.search(r"kTileMaxRows = (.*);", src).group(1))
    assert most * 4 < 1 << 32
    for cus in (32, 128, 256, 304):
        for N in [most - d for d in (0, 1, 15, 16, 17, 12288, 1 << 20)] + [1 << 29, 1 << 28]:
            ntiles = -(-N // 16)
            blocks = 3 * cus * -(-ntiles // (12 * cus))
            P = -(-ntiles // blocks)
            fewest = -(-ntiles // P)
            assert P <= 4 and max(blocks, fewest) * 256 < 1 << 32


@pytest.mark.parametrize("stages", [1, 3, 4, 7, 28, 32, 147, 148, 300])
@pytest.mark.parametrize("S", [4, 8])
@pytest.mark.parametrize("turns", [True, False])
def test_stages(stages, S, turns):
    seen = []
    for w in range(S):
        k0 = w if turns else w * stages // S
        n = (stages - w + S - 1) // S if turns else (w + 1) * stages // S - k0
        seen += [k0 + t * (S if turns else 1) for t in range(n)]
    assert sorted(seen) == list(range(stages))


@pytest.mark.parametrize("G", [1, 3, 4, 5, 28, 33, 112, 148, 255, 256])
@pytest.mark.parametrize("P", [1, 3, 6])
def test_metadata_items(G, P):
    chunks = (G + 3) // 4 if G > 8 else 2
    mul = -(-(1 << 32) // chunks)
    assert mul < 1 << 32
    rows, stride = 16 * P, 16 * P + 1
    words = set()
    for i in range(rows * chunks):
        r = (i * mul) >> 32
        assert r == i // chunks
        c = i - r * chunks
        words |= {(4 * c + g) * stride + r for g in range(4)}
    assert len(words) == 4 * rows * chunks and max(words) < 4 * chunks * stride   # one writer each, within the region
    for kb in range(G):                                      # what a wave reads: its tiles' rows of group kb
        assert all(kb * stride + r in words for r in range(rows))


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "int4"])
def test_lds_layouts(fmt):
    cols, row_bytes = {"bf16": (64, 128), "fp8": (128, 128), "int4": (128, 64)}[fmt]
    w_at = ((lambda r, p: r * 128 + ((p ^ (r & 7)) << 4)) if row_bytes == 128
            else (lambda r, p: r * 64 + ((p ^ ((r >> 1) & 3)) << 4)))
    x_at = lambda r, p: r * 2 * cols + ((p ^ (r & 7)) << 4)
    pieces, per_load = row_bytes // 16, 64 // (row_bytes // 16)
    lds = {}
    for i in range(row_bytes * 16 // 1024):                  # load i, lane l: row i*per_load + l/pieces, piece l%pieces
        for l in range(64):
            lds[w_at(i * per_load + l // pieces, l % pieces)] = (i * per_load + l // pieces, l % pieces)
    assert len(lds) == 16 * pieces and max(lds) < 16 * row_bytes
    for i in range(row_bytes // 64):
        for lane in range(64):
            assert lds[w_at(lane & 15, 4 * i + (lane >> 4))] == (lane & 15, 4 * i + (lane >> 4))
    xl = {x_at(m, p): (m, p) for m in range(16) for p in range(cols // 8)}
    assert len(xl) == 16 * cols // 8
    for j in range(cols // 32):
        for h in range(4):
            piece = 4 * j + h if fmt == "bf16" else (8 * (j >> 1) + 2 * h + (j & 1) if fmt == "fp8" else 4 * h + j)
            assert 8 * piece == step_col(fmt, j, h)          # x's 8 columns = the weights' of that lane group and step
    for p in range(4):                                       # 8 consecutive rows' same piece: 8 different 16-byte banks
        assert len({w_at(r, p) % 128 for r in range(8)}) == 8 and len({x_at(r, p) % 128 for r in range(8)}) == 8


@pytest.mark.parametrize("rem", range(0, 128, 16))
@pytest.mark.parametrize("row_bytes", [128, 1024, 1280])
@pytest.mark.parametrize("splits", [4, 8])
def test_ring_gives_every_stage_its_bytes(rem, row_bytes, splits):
    """Rows of any 16-byte remainder read line by line: the line a lane loads, where it puts it in the two-line ring and where
    a stage reads it, as the kernel computes them, give each stage its own 128 bytes of the row (zero past the row's end),
    from offsets inside the tile, with the 16 rows' pieces in 16 different bank groups."""
    rb = row_bytes + rem
    rng = np.random.default_rng(rb)
    tile = rng.integers(1, 256, 16 * rb, dtype=np.uint8)
    stages = -(-rb // 128)
    for split in range(splits):
        k0 = split * stages // splits
        n = (split + 1) * stages // splits - k0
        ring = np.zeros((16, 16, 16), np.uint8)           # row, piece, byte
        for t in range(n + 1 if n else 0):
            for lane in range(64):
                piece, r8 = lane % 8, lane // 8
                ws = (r8 * rb) & 127
                kb = k0 + t - 1
                inside = piece * 16 - ws < rb - (kb + 1) * 128
                off = r8 * rb - ws + piece * 16 + (kb + 1) * 128
                for i in range(2):
                    at = off + 8 * rb * i
                    assert not inside or 0 <= at <= 16 * rb - 16
                    put = (piece + r8 - (ws >> 4) + 8 * i + 8 * (t & 1)) & 15
                    ring[8 * i + r8, put] = tile[at:at + 16] if inside else 0
            if t == 0:
                continue
            for q in range(8):
                gets = [(q + row + 8 * ((t + 1) & 1)) & 15 for row in range(16)]
                assert len(set(gets)) == 16
                for row in range(16):
                    lo = (k0 + t - 1) * 128 + q * 16
                    want = tile[row * rb + lo:row * rb + lo + 16] if lo < rb else np.zeros(16, np.uint8)
                    assert np.array_equal(ring[row, gets[row]], want), (split, t, row, q)


def e4m3(b):                                              # codes 0..15: subnormals and the first binade
    return b * 2.0 ** -9 if b < 8 else (1 + (b - 8) / 8) * 2.0 ** -6


def test_int4_nibbles_as_e4m3():
    """All 16 codes in every position of a word: the byte pairs taken as e4m3, times 2^-2, are q 2^-11 in the order in which
    the activations are re-paired, so that a group's products are its weights' own."""
    order = [0, 2, 4, 6, 1, 3, 5, 7]                      # columns of a step's four bf16 pairs (i4_pair_x)
    perm = lambda hi, lo, sel: [(lo + hi)[k] for k in sel]
    x = np.arange(8)
    pairs = [x[0:2].tolist(), x[2:4].tolist(), x[4:6].tolist(), x[6:8].tolist()]
    paired = (perm(pairs[1], pairs[0], [0, 2]) + perm(pairs[3], pairs[2], [0, 2]) +
              perm(pairs[1], pairs[0], [1, 3]) + perm(pairs[3], pairs[2], [1, 3]))
    assert paired == order
    for word in [int("".join(f"{(q + 5 * j) % 16:x}" for j in range(8)), 16) for q in range(16)]:
        lo, hi = word & 0x0F0F0F0F, (word >> 4) & 0x0F0F0F0F
        got = [e4m3((h >> (8 * b)) & 0xFF) * 0.25 for h in (lo, hi) for b in range(4)]
        assert got == [((word >> (4 * c)) & 15) * 2.0 ** -11 for c in order]


def test_int4_powers_of_two():
    """Nibbles and sums of x at 2^-11, scales at 2^4, the finished sums times 2^7: the powers cancel, no group of finite
    activations leaves fp32, and products of the smallest activations are exact in it. Asymmetric scales keep every bit in
    the metadata word, those too large for the 2^4 with it on the nibbles and the zero point."""
    f32max, xmax, xmin = (2 - 2.0 ** -23) * 2.0 ** 127, (2 - 2.0 ** -7) * 2.0 ** 127, 2.0 ** -133
    assert np.array([0x3A00 << 16], np.uint32).view(np.float32)[0] == 2.0 ** -11
    assert 128 * 15 * 2.0 ** -11 * xmax < f32max and xmin * 2.0 ** -11 >= 2.0 ** -149
    s16 = np.arange(1 << 16, dtype=np.uint32)             # every bf16
    s16 = s16[(s16 & 0x7F80) != 0x7F80]
    s = (s16 << 16).view(np.float32).astype(np.float64)
    big = (s16 & 0x7F80) >= 0x7D80
    with np.errstate(over="ignore"):
        up = ((s16 << 16).view(np.float32) * np.float32(16)).view(np.uint32)
    assert not np.any(up[~big] & 0xFFFF)
    for z in (0, 5, 15):
        word = np.where(big, s16 << 16 | 129 << 8 | z << 4, up | 125 << 8 | z)
        scale = (word & 0xFFFF0000).astype(np.uint32).view(np.float32).astype(np.float64)
        factor = 2.0 ** (((word << 15 >> 23) & 0xFF).astype(np.int64) - 127)
        assert np.isfinite(scale).all()
        assert np.array_equal(scale * factor * 2.0 ** -9 * 2.0 ** 7, s)                      # on the nibbles
        assert np.array_equal(scale * (word & 0xFF) * 2.0 ** -11 * 2.0 ** 7, s * z)          # on the sums of x
