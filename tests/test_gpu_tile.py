"""GPU parity of the tile kernel (gemv_tile.h: the small-batch entry points with the variant left to the library) against
the CPU oracle, at the edges of its launch rule: one to six tiles of 16 rows per wave and more than one round of blocks,
rows that end inside a tile and inside a stage, one stage for many waves, long K, odd group counts, and metadata that is not
aligned for the wide loads. Bars as for the other small-batch kernels (test_gpu_batch.py)."""
import numpy as np
import pytest
import torch

from gpu_util import make, note
from paia_bench.inputs import to_device
from test_gpu_batch import check_rows, oracle_rows, run_batch, x_rows, xbits

pytestmark = pytest.mark.gpu

# (N, K / the format's K step, M): tiles on a 256-CU GPU 1, 2, 256, 257, 700, 1100, 1300, 1600 and 3200
EDGES = [(1, 1, 16), (17, 3, 3), (33, 9, 5), (4096, 5, 9), (4097, 2, 16), (11200, 3, 4), (17593, 2, 8), (20800, 1, 16),
         (25600, 3, 6), (51200, 1, 3), (48, 130, 16), (70, 67, 7), (20800, 21, 4)]
STEP = {"bf16": 72, "fp8": 144, "int4": 128, "int4zp": 128}   # BF16 and FP8: stages of 64 and 128 columns with a tail


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "int4", "int4zp"])
@pytest.mark.parametrize("N,kq,M", EDGES)
def test_edges(oracle, gemv_lib, cuda, fmt, N, kq, M):
    K = STEP[fmt] * kq
    ops, np_ops = make(fmt, N, K, bias=fmt != "int4")
    dev = to_device(ops, cuda)
    x = x_rows(M, K, 6000 + M + N + K)
    rows = np.unique(np.concatenate([np.arange(0, N, max(1, N // 150)), np.arange(max(0, N - 17), N)])).astype(np.int64)
    refs = oracle_rows(oracle, fmt, np_ops, xbits(x), rows)
    note(f"tile {fmt} M={M} N={N} K={K}")
    buf = torch.full((M * N + 64,), float("nan"), dtype=torch.bfloat16, device=cuda)
    y = run_batch(gemv_lib, fmt, dev, x.to(cuda), y=buf[:M * N].view(M, N))
    torch.cuda.synchronize()
    assert not torch.isnan(y).any() and torch.isnan(buf[M * N:]).all()
    check_rows(oracle, y, refs, f"tile {fmt} M={M} {N}x{K}", rows)


@pytest.mark.parametrize("fmt", ["int4", "int4zp"])
@pytest.mark.parametrize("off", [0, 2, 6, 8])
def test_metadata_alignment(gemv_lib, cuda, fmt, off):
    """Scales and zero points at any alignment of the contract (2 bytes and 1): bit for bit the aligned call's result."""
    N, K, M = 4112, 1024, 8
    ops, _ = make(fmt, N, K)
    dev = to_device(ops, cuda)
    x = x_rows(M, K, 77).to(cuda)
    note(f"tile metadata {fmt} offset {off}")
    want = run_batch(gemv_lib, fmt, dev, x)
    moved = dict(dev)
    s = torch.zeros(dev["scales"].numel() + 8, dtype=dev["scales"].dtype, device=cuda)
    moved["scales"] = s[off // 2: off // 2 + dev["scales"].numel()].copy_(dev["scales"].view(-1)).view(dev["scales"].shape)
    if fmt == "int4zp":
        z = torch.zeros(dev["zeros"].numel() + 16, dtype=torch.uint8, device=cuda)
        o = off + (off == 6)   # an odd address too
        moved["zeros"] = z[o: o + dev["zeros"].numel()].copy_(dev["zeros"].view(-1)).view(dev["zeros"].shape)
    got = run_batch(gemv_lib, fmt, moved, x)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "int4", "int4zp"])
def test_replays_and_rows(gemv_lib, cuda, fmt):
    """Captured and replayed with eager work between the replays, and with other activation rows beside it: every result
    bit for bit the eager one (the split order is fixed and a row does not depend on its neighbours)."""
    N, K, M = 6150, 2048, 12
    ops, _ = make(fmt, N, K, bias=fmt != "int4")
    dev = to_device(ops, cuda)
    x = x_rows(M, K, 9).to(cuda)
    note(f"tile replays {fmt}")
    eager = run_batch(gemv_lib, fmt, dev, x)
    torch.cuda.synchronize()
    x2 = torch.cat([x[:9], x_rows(7, K, 10).to(cuda) * 100]).contiguous()
    y2 = run_batch(gemv_lib, fmt, dev, x2)
    torch.cuda.synchronize()
    assert torch.equal(y2[:9].view(torch.int16), eager[:9].view(torch.int16))
    y = torch.empty_like(eager)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run_batch(gemv_lib, fmt, dev, x, y=y)
    for i in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), eager.view(torch.int16)), f"replay {i}"
        run_batch(gemv_lib, fmt, dev, x2)
        torch.cuda.synchronize()


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "int4", "int4zp"])
@pytest.mark.parametrize("M", [9, 16])
def test_rows_of_infinities_and_nan(gemv_lib, cuda, fmt, M):
    """Activation rows that hold infinities and NaN beside finite ones: not finite themselves, and every other row keeps its
    bits."""
    N, K = 2070, 1152
    ops, _ = make(fmt, N, K, bias=fmt != "int4")
    dev = to_device(ops, cuda)
    x = x_rows(M, K, 41).to(cuda)
    note(f"tile rows of infinities {fmt} M={M}")
    want = run_batch(gemv_lib, fmt, dev, x)
    bad = x.clone()
    bad[1, 5], bad[4, K - 1], bad[M - 1, 700] = float("inf"), float("nan"), float("-inf")
    y = run_batch(gemv_lib, fmt, dev, bad)
    torch.cuda.synchronize()
    keep = [m for m in range(M) if m not in (1, 4, M - 1)]
    assert torch.equal(y[keep].view(torch.int16), want[keep].view(torch.int16))
    # a weight of zero times an infinity is a NaN: no output of these rows is finite
    assert not torch.isfinite(y[[1, 4, M - 1]]).any()


@pytest.mark.parametrize("fmt", ["int4", "int4zp"])
@pytest.mark.parametrize("N,K,M", [(33, 262144, 16), (16, 300032, 3)])
def test_metadata_beyond_the_lds(oracle, gemv_lib, cuda, fmt, N, K, M):
    """Rows whose scales and zero points do not fit the block's LDS even for one tile (above K = 230912 at M = 16, 277504 at
    M <= 4): the call goes to the variant table's kernel."""
    ops, np_ops = make(fmt, N, K)
    x = x_rows(M, K, 43)
    note(f"tile metadata beyond LDS {fmt} M={M} {N}x{K}")
    dev = to_device(ops, cuda)
    y = run_batch(gemv_lib, fmt, dev, x.to(cuda))
    want = run_batch(gemv_lib, fmt, dev, x.to(cuda), gemv_lib.batch_pick_variant(fmt, M, N, K))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    check_rows(oracle, y, oracle_rows(oracle, fmt, np_ops, xbits(x)), f"{fmt} M={M} {N}x{K}")


@pytest.mark.parametrize("fmt", ["int4", "int4zp"])
@pytest.mark.parametrize("lo,hi", [(-125, -112), (-120, -55), (-50, 50), (60, 99), (100, 120)])
def test_int4_extreme_x(oracle, gemv_lib, cuda, fmt, lo, hi):
    """Activations over the whole bf16 range, rows of one call 2^5 apart, down to where the scaled products are subnormal and up to
    where a group's sum of q x alone would leave fp32 (scales are divided so that the output does not): gated as the
    reference gates."""
    N, K, M = 321, 640, 5
    ops, np_ops = make(fmt, N, K)
    if hi > 99:   # 15 * 640 * 2^120 alone is beyond fp32; with scales below 2^-14 the outputs are not
        ops["scales"] = (ops["scales"].float() * 2.0 ** -9).to(ops["scales"].dtype)
        np_ops["scales"] = ops["scales"].view(torch.int16).numpy().view(np.uint16)
    g = torch.Generator().manual_seed(lo * 1000 + hi)
    e = torch.randint(lo, hi + 1, (K,), generator=g).double()
    x0 = (1 + torch.rand(K, generator=g).double()) * torch.sign(torch.randn(K, generator=g).double()) * 2.0 ** e
    x = torch.stack([x0 * 2.0 ** (5 * m * (1 if hi < 60 or hi > 99 and m < 2 else -1)) for m in range(M)]).to(torch.bfloat16)
    note(f"tile extreme {fmt} {lo}..{hi}")
    y = run_batch(gemv_lib, fmt, to_device(ops, cuda), x.to(cuda))
    torch.cuda.synchronize()
    for m, (r64, _) in enumerate(oracle_rows(oracle, fmt, np_ops, xbits(x))):
        got = y[m].float().cpu().numpy().astype(np.float64)
        assert np.isfinite(r64).all() and np.isfinite(got).all(), (m, np.abs(r64).max())
        assert np.abs(got - r64).max() / np.abs(r64).max() < 2e-2, m


@pytest.mark.parametrize("fmt", ["int4", "int4zp"])
@pytest.mark.parametrize("M", [5, 16])
def test_int4_smallest_outputs(oracle, gemv_lib, cuda, fmt, M):
    """Outputs in bf16's subnormal range carry the error of their rounding and no more. The fp32 sums move in steps of 2^-142
    there: over the 32 groups of K = 4096 that adds 32 / 12 * 2^-284 to the rounding's variance 2^-266 / 12, a relative 1.2e-4
    (sums in steps of 2^-138 would add 3%)."""
    N, K = 2064, 4096
    ops, np_ops = make(fmt, N, K)
    x = (x_rows(M, K, 31).double() * 2.0 ** -129).to(torch.bfloat16)
    note(f"tile smallest outputs {fmt} M={M}")
    y = run_batch(gemv_lib, fmt, to_device(ops, cuda), x.to(cuda)).float().cpu().numpy().astype(np.float64)
    want = np.stack([r for r, _ in oracle_rows(oracle, fmt, np_ops, xbits(x))])
    assert 2.0 ** -130 < np.sqrt((want ** 2).mean()) and np.abs(want).max() < 2.0 ** -125
    rounding = np.rint(want * 2.0 ** 133) * 2.0 ** -133 - want
    assert np.sqrt(((y - want) ** 2).mean() / (rounding ** 2).mean()) < 1.005


def test_int4zp_largest_scales(oracle, gemv_lib, cuda):
    """One group with a scale of 2^124: its row is right, and every other row of the call keeps its bits. An infinite scale
    stays in its row too."""
    N, K, M = 4112, 1024, 6
    ops, np_ops = make("int4zp", N, K)
    dev = to_device(ops, cuda)
    x = (x_rows(M, K, 32).double() * 2.0 ** -12).to(torch.bfloat16)
    xd = x.to(cuda)
    note("tile largest scales int4zp")
    want = run_batch(gemv_lib, "int4zp", dev, xd)
    scales = ops["scales"].clone()
    scales[100, 3] = 2.0 ** 124
    big = dict(dev, scales=scales.to(cuda))
    y = run_batch(gemv_lib, "int4zp", big, xd)
    np_big = dict(np_ops, scales=scales.view(torch.int16).numpy().view(np.uint16))
    rows = np.array([100], dtype=np.int64)
    check_rows(oracle, y, oracle_rows(oracle, "int4zp", np_big, xbits(x), rows), "row 100", rows)
    keep = torch.arange(N, device=cuda) != 100
    assert torch.equal(y[:, keep].view(torch.int16), want[:, keep].view(torch.int16))
    scales[100, 3] = float("inf")
    y = run_batch(gemv_lib, "int4zp", dict(dev, scales=scales.to(cuda)), xd)
    assert not torch.isfinite(y[:, 100]).any()
    assert torch.equal(y[:, keep].view(torch.int16), want[:, keep].view(torch.int16))


# BF16 and FP8 row lengths: whole 128-byte lines, then every remainder of 16 bytes, read line by line (N = 528: one tile per
# block, 4112 and 13000: two and four tiles per wave) or, for short rows, split; M past what the row-streaming kernel takes
@pytest.mark.parametrize("fmt", ["bf16", "fp8"])
@pytest.mark.parametrize("N,row_bytes,M", [(528, 8192, 9), (4112, 2048, 16), (528, 8208, 16), (531, 8320 - 16, 9),
                                           (4112, 1280 + 16, 16), (4112, 1280 + 32, 8), (4100, 4096 + 48, 11),
                                           (4112, 2048 + 64, 9), (13000, 1408 + 80, 16), (8200, 2176 - 32, 8),
                                           (4112, 1024 + 112, 16), (528, 1024 + 80, 12), (1041, 2400 + 16, 9), (8200, 16, 9), (4112, 9200, 8)])
def test_row_forms(oracle, gemv_lib, cuda, fmt, N, row_bytes, M):
    row_form(oracle, gemv_lib, cuda, fmt, N, row_bytes, M)


# The same with four activation rows staged: line by line with three and seven tiles per wave, as a block per tile, and
# in 8-wave blocks
@pytest.mark.parametrize("fmt,N,row_bytes,M", [("fp8", 12000, 3600, 3), ("fp8", 12001, 3600, 4), ("fp8", 25000, 2000, 4),
                                               ("fp8", 17000, 5008, 4), ("bf16", 9001, 16400, 4)])
def test_row_forms_few_rows(oracle, gemv_lib, cuda, fmt, N, row_bytes, M):
    row_form(oracle, gemv_lib, cuda, fmt, N, row_bytes, M)


def row_form(oracle, gemv_lib, cuda, fmt, N, row_bytes, M):
    """Also from weights 16 bytes past a line (bit for bit the same), and with a row of NaN between finite ones: rows that share
    its lines keep their results."""
    K = row_bytes // (2 if fmt == "bf16" else 1)
    ops, np_ops = make(fmt, N, K, bias=True)
    dev = to_device(ops, cuda)
    x = x_rows(M, K, 8000 + M + N + K)
    rows = np.unique(np.concatenate([np.arange(0, N, max(1, N // 100)), np.arange(max(0, N - 17), N)])).astype(np.int64)
    refs = oracle_rows(oracle, fmt, np_ops, xbits(x), rows)
    note(f"tile row forms {fmt} M={M} N={N} row bytes {row_bytes}")
    x = x.to(cuda)
    y = run_batch(gemv_lib, fmt, dev, x)
    torch.cuda.synchronize()
    check_rows(oracle, y, refs, f"tile {fmt} M={M} {N}x{K}", rows)
    name = "W" if fmt == "bf16" else "Wq"
    w = dev[name].contiguous().view(torch.uint8).view(-1)
    room = torch.empty(w.numel() + 16, dtype=torch.uint8, device=cuda)
    room[16:].copy_(w)
    moved = dict(dev)
    moved[name] = room[16:].view(dev[name].dtype).view(dev[name].shape)
    y2 = run_batch(gemv_lib, fmt, moved, x)
    torch.cuda.synchronize()
    assert torch.equal(y2.view(torch.int16), y.view(torch.int16))
    bad = torch.arange(5, N, 7, device=cuda)
    room[16:].view(N, row_bytes)[bad] = 0x7F if fmt == "fp8" else 0xFF   # e4m3 and bf16 NaN
    y3 = run_batch(gemv_lib, fmt, moved, x)
    torch.cuda.synchronize()
    assert torch.isnan(y3[:, bad]).all()
    keep = torch.ones(N, dtype=torch.bool, device=cuda)
    keep[bad] = False
    assert torch.equal(y3[:, keep].view(torch.int16), y[:, keep].view(torch.int16))


# Both sides of the rule that keeps a call on the variant table's kernel: (format, M, N, K, on the table's kernel). On the
# tile kernel's side only calls of 10^5 outputs, enough for some to differ.
ROUTES = [("bf16", 8, 592, 3592, True), ("bf16", 8, 350, 9712, True), ("bf16", 8, 64, 6936, True),
          ("bf16", 6, 18428, 1872, True), ("bf16", 5, 19230, 1864, True), ("bf16", 6, 19230, 2104, False),
          ("bf16", 5, 14106, 8192, True), ("bf16", 4, 14106, 8256, True), ("bf16", 4, 17000, 8192, False),
          ("bf16", 8, 10000, 8192, False), ("bf16", 8, 14106, 8320, False), ("fp8", 3, 43820, 3696, True),
          ("fp8", 3, 36392, 2160, False), ("fp8", 3, 12264, 16256, True), ("fp8", 5, 12264, 16256, False),
          ("fp8", 7, 74000, 528, True), ("fp8", 7, 73000, 528, False), ("fp8", 9, 74000, 528, False),
          ("int4", 2, 629, 18048, True), ("int4zp", 2, 629, 18048, True), ("int4", 2, 17000, 7552, True),
          ("int4zp", 2, 17000, 6016, False), ("int4zp", 2, 25000, 6016, True),
          ("int4zp", 2, 25000, 5504, False),
          ("int4", 2, 28672, 4096, True), ("int4", 2, 20000, 4096, False), ("int4", 3, 1400, 3968, True),
          ("bf16", 8, 1024, 4096, True),
          # six tiles per wave: metadata beyond the LDS above K = 37376
          ("int4", 16, 24576, 38400, True), ("int4zp", 16, 24576, 37376, False)]


@pytest.mark.parametrize("fmt,M,N,K,table", ROUTES)
def test_route(gemv_lib, cuda, fmt, M, N, K, table):
    """Where the table's kernel is the faster one a default call gives its bits; elsewhere the tile kernel's sums, split
    over a block's waves, round another way somewhere. Both are within twice the rounding of bf16."""
    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the bounds are in tiles per CU: these sizes are for 256")
    g = torch.Generator(device=cuda).manual_seed(N + K)
    dev = {"N": N}
    if fmt == "bf16":
        dev["W"] = torch.randn(N, K, dtype=torch.bfloat16, device=cuda, generator=g)
    elif fmt == "fp8":
        dev["Wq"] = torch.randint(0, 0x78, (N, K), dtype=torch.uint8, device=cuda, generator=g)
        dev["scale"] = torch.rand(N, device=cuda, generator=g)
    else:
        dev["Wq"] = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=cuda, generator=g)
        dev["scales"] = torch.rand(N, K // 128, device=cuda, generator=g).to(
            torch.float16 if fmt == "int4" else torch.bfloat16)
        dev["zeros"] = torch.randint(0, 256, (N, (K // 128 + 1) // 2), dtype=torch.uint8, device=cuda, generator=g)
    x = x_rows(M, K, 11).to(cuda)
    note(f"route {fmt} M={M} {N}x{K}")
    y = run_batch(gemv_lib, fmt, dev, x)
    want = run_batch(gemv_lib, fmt, dev, x, gemv_lib.batch_pick_variant(fmt, M, N, K))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), want.view(torch.int16)) == table
    d = (y.float() - want.float()).norm() / want.float().norm()
    assert d < 2.0 ** -8
