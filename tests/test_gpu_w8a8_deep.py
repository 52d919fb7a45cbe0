"""The many-row W8A8 / W4A8 kernel (prompt chunks), which eager calls with automatic tiles run past
128 rows: every tile it has, at ragged M, N and K, bit for bit against the formula in 64-bit sums
(the INT32 sums are exact and the epilogue's roundings are fixed: fp32 after each scale, then fp16).
"""
import pytest
import torch

import kernels as K
from gpu_util import note
from specq import gen
from specq.plan import Plan

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(fmt, M, N, Kd, seed):
    """(activations, token scales, packed weight, channel scales, the weight's integers)."""
    a, sa = (t.to(DEV) for t in gen.w8a8_acts(M, Kd, seed=seed))
    g = torch.Generator(device=DEV).manual_seed(seed)
    sw = torch.rand(N, device=DEV, generator=g) * 1e-3 + 1e-4
    if fmt == "w8a8":
        w = torch.randint(-127, 128, (N, Kd), dtype=torch.int8, device=DEV, generator=g)
        return a, sa, K.pack_weight_int8(w), sw, w
    q = torch.randint(0, 16, (N, Kd), dtype=torch.uint8, device=DEV, generator=g)
    half = Kd // 2
    return a, sa, K.pack_weight_w4a8((q[:, :half] | (q[:, half:] << 4)).contiguous()), sw, q.to(torch.int8) - 8


def formula(a, sa, w, sw):
    acc = (a.double() @ w.double().t()).float()
    return ((acc * sa[:, None]) * sw[None, :]).half()


# (format, M, N, K, kernel): one row past a tile, one short of it, odd N (unaligned output rows), K a
# partial step, an odd number of steps, fewer steps than the ring holds.
CASES = [
    ("w8a8", 150, 10001, 3088, "deep_kernel<2, 4, 3, 1>"),
    ("w8a8", 193, 7001, 1104, "deep_kernel<2, 4, 3, 1>"),
    ("w8a8", 513, 3001, 1040, "deep_kernel<2, 4, 3, 1>"),
    ("w8a8", 385, 7001, 1104, "deep_kernel<4, 4, 4, 1>"),
    ("w8a8", 300, 10001, 3088, "deep_kernel<4, 4, 4, 1>"),
    ("w8a8", 641, 10001, 3088, "deep_kernel<4, 4, 2, 1>"),
    ("w8a8", 1281, 28673, 208, "deep_kernel<4, 4, 2, 1>"),
    ("w8a8", 1281, 10001, 3088, "deep_mix_kernel<1>"),    # whole tiles only
    ("w8a8", 1537, 28673, 1104, "deep_mix_kernel<1>"),    # three rounds of them, then halves
    ("w8a8", 897, 15000, 144, "deep_mix_kernel<1>"),
    ("w4a8", 700, 10001, 3088, "deep_kernel<4, 4, 2, 2>"),
    ("w4a8", 193, 28673, 208, "deep_kernel<4, 4, 2, 2>"),
    ("w4a8", 1023, 3001, 1040, "deep_kernel<4, 4, 2, 2>"),
]


@pytest.mark.parametrize("fmt, M, N, Kd, name", CASES)
def test_many_rows_bit_exact(fmt, M, N, Kd, name):
    note(f"{fmt} many rows M={M} N={N} K={Kd}")
    a, sa, wp, sw, w = operands(fmt, M, N, Kd, seed=M)
    mm = K.w8a8_matmul if fmt == "w8a8" else K.w4a8_matmul
    big = torch.full((M + 3, N + 5), 7.0, dtype=torch.float16, device=DEV)
    _, ck = mm(a, sa, wp, sw, out=big[:M, :N], BLOCK_M=None)
    torch.cuda.synchronize()
    assert name in ck.name, ck.name
    assert torch.equal(big[:M, :N].view(torch.int16), formula(a, sa, w, sw).view(torch.int16)), ck.name
    assert bool((big[M:] == 7.0).all()) and bool((big[:, N:] == 7.0).all()), "stored past M or N"


# Every tile, the mixed kernel's halves among them, at output rows that lanes store 16 bytes at a time:
# contiguous ones, and padded ones whose last pieces are stored value by value.
@pytest.mark.parametrize("fmt, M, N, Kd, name", [
    ("w8a8", 150, 10000, 3088, "deep_kernel<2, 4, 3, 1>"),
    ("w8a8", 385, 7000, 1104, "deep_kernel<4, 4, 4, 1>"),
    ("w8a8", 641, 10000, 3088, "deep_kernel<4, 4, 2, 1>"),
    ("w8a8", 1281, 10000, 3088, "deep_mix_kernel<1>"),
    ("w8a8", 1023, 8184, 1040, "deep_mix_kernel<1>"),   # halves only
    ("w4a8", 700, 10000, 3088, "deep_kernel<4, 4, 2, 2>"),
])
@pytest.mark.parametrize("odd", [0, 1, 5])
def test_many_rows_aligned_output_rows(fmt, M, N, Kd, name, odd):
    N -= odd
    note(f"{fmt} many rows, aligned output rows M={M} N={N} K={Kd}")
    a, sa, wp, sw, w = operands(fmt, M, N, Kd, seed=M + 1)
    mm = K.w8a8_matmul if fmt == "w8a8" else K.w4a8_matmul
    big = torch.full((M + 3, N + odd + (8 if odd else 0)), 7.0, dtype=torch.float16, device=DEV)
    _, ck = mm(a, sa, wp, sw, out=big[:M, :N], BLOCK_M=None)
    torch.cuda.synchronize()
    assert name in ck.name and big.stride(0) % 8 == 0, (ck.name, big.stride(0))
    assert torch.equal(big[:M, :N].view(torch.int16), formula(a, sa, w, sw).view(torch.int16)), ck.name
    assert bool((big[M:] == 7.0).all()) and bool((big[:, N:] == 7.0).all()), "stored past M or N"


@pytest.mark.parametrize("M", [1, 129, 400])
def test_many_rows_of_a_larger_grid(M):
    """grid_m_max without a plan: the launch covers rows that there are not, whose workgroups end at once.
    (No rows at all: an empty tensor has a null pointer, which the library refuses.)"""
    note(f"many rows M={M} grid_m_max=1281")
    a, sa, wp, sw, w = operands("w8a8", M, 10000, 3088, seed=9)
    out = torch.full((1281, 10000), 7.0, dtype=torch.float16, device=DEV)
    _, ck = K.w8a8_matmul(a[:M], sa[:M], wp, sw, out=out[:M], BLOCK_M=None, grid_m_max=1281)
    torch.cuda.synchronize()
    assert "deep_mix_kernel<1>" in ck.name, ck.name
    assert torch.equal(out[:M].view(torch.int16), formula(a[:M], sa[:M], w, sw).view(torch.int16))
    assert bool((out[M:] == 7.0).all())


def test_many_rows_grouped_members():
    """Members whose widths are no whole tiles, one below a tile, on a strided activation."""
    M, Kd, Ns = 1400, 1104, (7001, 40, 5000, 3000)
    note(f"grouped many rows M={M} N={Ns} K={Kd}")
    ops = [operands("w8a8", M, N, Kd, seed=900 + i) for i, N in enumerate(Ns)]
    wide = torch.zeros((M, Kd + 48), dtype=torch.int8, device=DEV)
    wide[:, 16:16 + Kd] = ops[0][0]
    outs, ck = K.w8a8_matmul_grouped(wide[:, 16:16 + Kd], ops[0][1], [(o[2], o[3]) for o in ops], BLOCK_M=None)
    torch.cuda.synchronize()
    assert "deep_" in ck.name, ck.name
    for o, op in zip(outs, ops):
        ref = formula(ops[0][0], ops[0][1], op[4], op[3])
        assert torch.equal(o.view(torch.int16), ref.view(torch.int16)), op[2].N


def test_plan_at_grid_tiles_of_many_rows():
    """plan_tiles="grid" asks for tiles that can be named explicitly: same bits, no row past M written."""
    M, N, Kd, active = 700, 7000, 1040, 601
    note(f"plan grid tiles M={M} active={active}")
    a, sa, wp, sw, w = operands("w8a8", M, N, Kd, seed=5)
    plan = Plan(DEV)
    plan.set(1, active)
    out = torch.full((M, N), 7.0, dtype=torch.float16, device=DEV)
    K.w8a8_matmul(a, sa, wp, sw, out=out, BLOCK_M=None, plan=plan.gemm, grid_m_max=M, plan_tiles="grid")
    torch.cuda.synchronize()
    assert torch.equal(out[:active].view(torch.int16), formula(a, sa, w, sw)[:active].view(torch.int16))
    assert bool((out[active:] == 7.0).all())


# (format, M, N, K, row stride in bytes, kernel): every tile height with a tile's rows spanning more than
# 4 GiB, the 64-row one also within it, the mixed launch as whole tiles and as halves.
WIDE = [
    ("w8a8", 193, 7001, 1104, 40 << 20, "deep_kernel<2, 4, 3, 1>"),
    ("w8a8", 193, 7001, 1104, 80 << 20, "deep_kernel<2, 4, 3, 1>"),
    ("w8a8", 385, 7001, 1104, 40 << 20, "deep_kernel<4, 4, 4, 1>"),
    ("w8a8", 641, 10001, 3088, 34 << 20, "deep_kernel<4, 4, 2, 1>"),
    ("w8a8", 513, 20000, 2048, 20 << 20, "deep_mix_kernel<1>"),
    ("w8a8", 1024, 8192, 1040, 34 << 20, "deep_mix_kernel<1>"),
    ("w4a8", 193, 28673, 208, 40 << 20, "deep_kernel<4, 4, 2, 2>"),
]


@pytest.mark.parametrize("fmt, M, N, Kd, ld, name", WIDE)
def test_many_rows_over_wide_strides(fmt, M, N, Kd, ld, name):
    """Activation rows that span gigabytes within a tile (one token of each long sequence): every row is
    read where it lies, far past the 32 bits of a buffer offset."""
    note(f"{fmt} many rows M={M} N={N} K={Kd} lda={ld}")
    a, sa, wp, sw, w = operands(fmt, M, N, Kd, seed=6)
    wide = torch.empty((M, ld), dtype=torch.int8, device=DEV)
    wide[:, :Kd] = a
    mm = K.w8a8_matmul if fmt == "w8a8" else K.w4a8_matmul
    out, ck = mm(wide[:, :Kd], sa, wp, sw, BLOCK_M=None)
    torch.cuda.synchronize()
    del wide
    torch.cuda.empty_cache()
    assert name in ck.name, ck.name
    assert torch.equal(out.view(torch.int16), formula(a, sa, w, sw).view(torch.int16)), ck.name


@pytest.mark.parametrize("fmt, M, N, Kd, ld, tile", [
    ("w8a8", 256, 8192, 8192, 40 << 20, {}),                      # a streaming tile by its price
    ("w8a8", 72, 4096, 4096, 64 << 20, {}),
    ("w8a8", 9, 4096, 4096, 300 << 20, {}),                       # 16-row tiles
    ("w8a8", 500, 3001, 1040, 20 << 20, dict(BLOCK_M=304)),       # explicit tiles, split K
    ("w8a8", 300, 1030, 1296, 20 << 20, dict(BLOCK_M=208, BLOCK_N=64, split_k=3)),
    ("w4a8", 144, 5120, 1040, 40 << 20, {}),
])
def test_streaming_tiles_over_wide_strides(fmt, M, N, Kd, ld, tile):
    """Rows further apart than the streaming kernels' offsets reach run a many-row kernel."""
    note(f"{fmt} wide strides M={M} N={N} K={Kd} lda={ld} {tile}")
    a, sa, wp, sw, w = operands(fmt, M, N, Kd, seed=16)
    wide = torch.empty((M, ld), dtype=torch.int8, device=DEV)
    wide[:, :Kd] = a
    mm = K.w8a8_matmul if fmt == "w8a8" else K.w4a8_matmul
    out, _ = mm(wide[:, :Kd], sa, wp, sw, **dict(dict(BLOCK_M=None), **tile))
    outs, _ = K.w8a8_matmul_grouped(wide[:, :Kd], sa, [(wp, sw), (wp, sw)], **dict(dict(BLOCK_M=None), **tile))
    torch.cuda.synchronize()
    del wide
    torch.cuda.empty_cache()
    ref = formula(a, sa, w, sw).view(torch.int16)
    for o in (out, *outs):
        assert torch.equal(o.view(torch.int16), ref)


@pytest.mark.parametrize("M, Ns", [(37500, (14336, 14336)), (70100, (5120, 5120, 5120))])
def test_many_rows_past_the_counter_region(M, Ns):
    """Grouped launches of more tiles than the split counters: the many-row kernel uses none."""
    Kd = 256
    note(f"w4a8 grouped many rows M={M} N={Ns} K={Kd}")
    ops = [operands("w4a8", M, N, Kd, seed=40 + i) for i, N in enumerate(Ns)]
    a, sa = ops[0][:2]
    outs, ck = K.w8a8_matmul_grouped(a, sa, [(o[2], o[3]) for o in ops], BLOCK_M=None)
    torch.cuda.synchronize()
    assert "deep_kernel<4, 4, 2, 2>" in ck.name, ck.name
    for o, op in zip(outs, ops):
        for rows in (slice(0, 300), slice(M // 2, M // 2 + 300), slice(M - 300, M)):
            ref = formula(a[rows], sa[rows], op[4], op[3])
            assert torch.equal(o[rows].view(torch.int16), ref.view(torch.int16)), rows


@pytest.mark.parametrize("block_m", [48, 64, 128, 208, 304])
@pytest.mark.parametrize("block_n, split_k", [(64, 1), (64, 3), (128, 1), (128, 4)])
def test_several_chunks_of_the_streaming_kernel(block_m, block_n, split_k):
    """Two and three M-chunks, the last ragged, whose weight loads stay in L2; one chunk keeps the other kind."""
    N, Kd = 1030, 1296
    note(f"w8a8 chunks BLOCK_M={block_m} BLOCK_N={block_n} split_k={split_k}")
    a, sa, wp, sw, w = operands("w8a8", 2 * block_m + 1, N, Kd, seed=block_m)
    kw = dict(BLOCK_M=block_m, BLOCK_N=block_n, split_k=split_k)
    for M, name in ((block_m, "w8a8_ws_kernel"), (block_m + 17, "chunks_ws_kernel"), (2 * block_m + 1, "chunks_ws_kernel")):
        out, ck = K.w8a8_matmul(a[:M], sa[:M], wp, sw, **kw)
        torch.cuda.synchronize()
        assert name in ck.name, (M, ck.name)
        assert torch.equal(out.view(torch.int16), formula(a[:M], sa[:M], w, sw).view(torch.int16)), (M, ck.name)


# Over distinct weights (a model's layers) the many-row kernel ran at 0.79 to 0.91 times the streaming
# kernel's speed at the first shapes, and faster at the last.
@pytest.mark.parametrize("variant, M, N, Kd, many", [(1, 256, 8192, 8192, False), (1, 178, 6400, 9760, False),
                                                     (1, 350, 5120, 5120, False), (2, 256, 13824, 5120, False),
                                                     (1, 1024, 8192, 8192, True), (2, 1024, 13824, 5120, True)])
def test_weights_from_memory_decide_the_kernel(variant, M, N, Kd, many):
    note(f"attrs variant={variant} M={M} N={N} K={Kd}")
    assert ("deep_" in K.KernelInfo(0, variant, M, N, Kd, 0, 0, 4, 0).name) == many
