"""The tile kernel's index arithmetic (paia-project_amd/csrc/gemv_tile.h) replayed on the CPU: every tile has one unit and
every stage one wave, the XCD order is a permutation, the metadata items divide exactly and stay in their LDS words, and the
swizzled LDS layouts bring each lane the columns its MFMA step takes, without a bank conflict among 8 rows."""
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
