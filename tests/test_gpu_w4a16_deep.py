"""The many-row W4A16 kernel (prompt chunks) against the streaming kernel it stands in for, bit for
bit (one fp32 summation order for every tile), and both against 64-bit sums.

Tolerance of the latter: the fp32 sums of K products and the fp16 rounding of the output, 2^-11 of
the value and K * 2^-24 of the sum of the products' magnitudes.
"""
import pytest
import torch

import kernels as K
from gpu_util import note

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(layout, M, N, Kd, group, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn((M, Kd), device=DEV, generator=g).half()
    q = torch.randint(0, 16, (N, Kd), dtype=torch.uint8, device=DEV, generator=g)
    sc = (torch.rand((N, Kd // group), device=DEV, generator=g) * 0.02 + 0.002).half()
    half = Kd // 2
    u8 = (q[:, :half] | (q[:, half:] << 4)).contiguous()
    wp = u8 if layout == "u8" else (K.pack_int4_i32(q) if layout == "i32" else K.pack_weight_int4(u8))
    deq = ((q.half() - 8).view(N, -1, group) * sc[..., None]).view(N, Kd)
    return a, wp, sc, deq


# (layout, M, N, K, group, split_k): one row past a tile and one short, odd N, an odd number of K
# blocks per stream and per split, a last split shorter than the others, one block in all.
CASES = [
    ("packed", 1024, 4096, 4096, 128, 0),
    ("packed", 1023, 4090, 1920, 128, 4),
    ("packed", 1023, 4001, 1664, 64, 5),
    ("packed", 1023, 4090, 2176, 128, 3),
    ("packed", 700, 4096, 4096, 4096, 0),
    ("packed", 1023, 4096, 640, 128, 2),
    ("i32", 895, 4100, 1792, 128, 4),
    ("i32", 1023, 4090, 1408, 32, 3),
    ("u8", 1000, 4096, 2304, 128, 4),
    ("u8", 769, 4030, 1280, 16, 4),
]


@pytest.mark.parametrize("layout, M, N, Kd, group, split_k", CASES)
def test_many_rows_bits_of_the_streaming_kernel(layout, M, N, Kd, group, split_k):
    note(f"w4a16 many rows {layout} M={M} N={N} K={Kd} group={group} split_k={split_k}")
    a, wp, sc, deq = operands(layout, M, N, Kd, group, seed=M)
    big = torch.full((M + 3, N + 8), 7.0, dtype=torch.float16, device=DEV)
    kw = dict(group=group, BLOCK_K=min(64, group), split_k=split_k)
    _, ck = K.w4a16_matmul(a, wp, sc, out=big[:M, :N], BLOCK_M=None, **kw)
    ws, ck2 = K.w4a16_matmul(a, wp, sc, BLOCK_M=128, **kw)
    torch.cuda.synchronize()
    assert "deep_kernel" in ck.name and "ws_kernel" in ck2.name, (ck.name, ck2.name)
    assert torch.equal(big[:M, :N].view(torch.int16), ws.view(torch.int16)), ck.name
    assert bool((big[M:] == 7.0).all()) and bool((big[:, N:] == 7.0).all()), "stored past M or N"
    ref, mag = a.double() @ deq.double().t(), a.double().abs() @ deq.double().abs().t()
    assert bool(((ws.double() - ref).abs() <= ref.abs() * 2.0 ** -11 + mag * Kd * 2.0 ** -24 + 1e-7).all())


@pytest.mark.parametrize("M", [1, 129, 400])
def test_many_rows_of_a_larger_grid(M):
    """grid_m_max without a plan: the launch covers rows that there are not, whose workgroups end at once.
    (No rows at all: an empty tensor has a null pointer, which the library refuses.)"""
    note(f"w4a16 many rows M={M} grid_m_max=1024")
    a, wp, sc, _ = operands("packed", M, 4096, 4096, 128, seed=10)
    out = torch.full((1024, 4096), 7.0, dtype=torch.float16, device=DEV)
    _, ck = K.w4a16_matmul(a[:M], wp, sc, out=out[:M], BLOCK_M=None, grid_m_max=1024)
    torch.cuda.synchronize()
    assert "deep_kernel" in ck.name, ck.name
    ref, _ = K.w4a16_matmul(a[:M], wp, sc, BLOCK_M=64)
    assert torch.equal(out[:M].view(torch.int16), ref.view(torch.int16))
    assert bool((out[M:] == 7.0).all())


def test_many_rows_grouped_and_nonfinite_rows():
    """Grouped members of unequal width; an activation row with Inf and NaN leaves the other rows alone."""
    M, Kd, Ns = 1020, 4096, (2048, 1030, 900)
    note(f"w4a16 grouped many rows M={M} N={Ns}")
    ops = [operands("packed", M, N, Kd, 128, seed=70 + i) for i, N in enumerate(Ns)]
    a = ops[0][0].clone()
    a[5, 3], a[5, 700], a[1019, 4095] = float("inf"), float("nan"), float("inf")
    outs, ck = K.w4a16_matmul_grouped(a, [(o[1], o[2]) for o in ops], split_k=4)
    torch.cuda.synchronize()
    assert "deep_kernel" in ck.name, ck.name
    for o, op in zip(outs, ops):
        ref, _ = K.w4a16_matmul(a, op[1], op[2], BLOCK_M=128, split_k=4)
        assert torch.equal(o.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("layout, M, N, Kd, ld", [("packed", 700, 4096, 4096, 12 << 20), ("packed", 700, 4096, 4096, 17 << 20),
                                                  ("u8", 385, 8192, 4096, 18 << 20), ("i32", 385, 8192, 4096, 40 << 20)])
def test_many_rows_over_wide_strides(layout, M, N, Kd, ld):
    """Activation rows that span more than 2 or 4 GiB within a tile: every row is read where it lies."""
    note(f"w4a16 many rows {layout} M={M} N={N} lda={ld}")
    a, wp, sc, _ = operands(layout, M, N, Kd, 128, seed=6)
    wide = torch.empty((M, ld), dtype=torch.float16, device=DEV)
    wide[:, :Kd] = a
    out, ck = K.w4a16_matmul(wide[:, :Kd], wp, sc, BLOCK_M=None)
    ref, _ = K.w4a16_matmul(a, wp, sc, BLOCK_M=128)
    torch.cuda.synchronize()
    del wide
    torch.cuda.empty_cache()
    assert "deep_kernel" in ck.name, ck.name
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("layout, M, N, Kd, ld, kw", [
    ("packed", 72, 4096, 4096, 17 << 20, {}),
    ("packed", 300, 6144, 1408, 10 << 20, dict(split_k=3)),              # 2 GiB and an odd number of blocks
    ("u8", 160, 1030, 1280, 16 << 20, dict(BLOCK_M=160, BLOCK_N=64)),
    ("i32", 9, 1030, 1280, 160 << 20, {}),
])
def test_streaming_tiles_over_wide_strides(layout, M, N, Kd, ld, kw):
    """Rows further apart than the streaming kernels' offsets reach run the many-row kernel; what lies
    between the rows (NaN here) is not read."""
    note(f"w4a16 wide strides {layout} M={M} N={N} lda={ld} {kw}")
    a, wp, sc, _ = operands(layout, M, N, Kd, 128, seed=17)
    wide = torch.full((M, ld), float("nan"), dtype=torch.float16, device=DEV)
    wide[:, :Kd] = a
    kw = dict(dict(BLOCK_M=None), **kw)
    out, _ = K.w4a16_matmul(wide[:, :Kd], wp, sc, **kw)
    outs, _ = K.w4a16_matmul_grouped(wide[:, :Kd], [(wp, sc), (wp, sc)], **kw)
    ref, _ = K.w4a16_matmul(a, wp, sc, **kw)
    torch.cuda.synchronize()
    del wide
    torch.cuda.empty_cache()
    for o in (out, *outs):
        assert torch.equal(o.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("members", [1, 2])
def test_many_rows_past_the_counter_region(members):
    """More tiles than there are split counters: the many-row kernel uses none."""
    M, N, Kd = 262500, 4096 // members, 4096
    note(f"w4a16 many rows M={M} members={members}")
    a = torch.randn((M, Kd), device=DEV, generator=torch.Generator(device=DEV).manual_seed(8)).half()
    ops = [operands("packed", 1, N, Kd, 128, seed=80 + i) for i in range(members)]
    if members == 1:
        out, ck = K.w4a16_matmul(a, *ops[0][1:3], BLOCK_M=None, split_k=4)
        outs = [out]
    else:
        outs, ck = K.w4a16_matmul_grouped(a, [o[1:3] for o in ops], split_k=4)
    torch.cuda.synchronize()
    assert "deep_kernel" in ck.name, ck.name
    for o, op in zip(outs, ops):
        for rows in (slice(0, 300), slice(M - 300, M)):
            ref, _ = K.w4a16_matmul(a[rows], *op[1:3], BLOCK_M=128, split_k=4)
            assert torch.equal(o[rows].view(torch.int16), ref.view(torch.int16)), rows


@pytest.mark.parametrize("block_m", [80, 96, 112, 128, 144, 160])
@pytest.mark.parametrize("layout, rows", [("packed", 1), ("packed", 161), ("u8", 17), ("i32", 40)])
def test_several_chunks_of_the_streaming_kernel(block_m, layout, rows):
    """Two and three M-chunks, the last ragged: the bits of 64-row tiles, whose weight loads are the other kind."""
    M, N, Kd = block_m + rows, 1030, 1280
    note(f"w4a16 chunks {layout} M={M} BLOCK_M={block_m}")
    a, wp, sc, _ = operands(layout, M, N, Kd, 128, seed=block_m)
    out, ck = K.w4a16_matmul(a, wp, sc, BLOCK_M=block_m)
    ref, ck64 = K.w4a16_matmul(a, wp, sc, BLOCK_M=64)
    torch.cuda.synchronize()
    assert "chunks_ws_kernel" in ck.name and "w4a16_ws_kernel" in ck64.name, (ck.name, ck64.name)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), ck.name


@pytest.mark.parametrize("kind, variant, M, N, Kd", [(0, 1, 513, 20000, 2048), (0, 2, 700, 10001, 3088), (1, 2, 1024, 4096, 4096)])
def test_streaming_tile_of_a_many_row_shape_names_itself(kind, variant, M, N, Kd):
    """`variant` | 32: a tile whose numbers, given back, ask for the same kernel."""
    note(f"attrs kind={kind} variant={variant} M={M} N={N} K={Kd}")
    assert "deep_" in K.KernelInfo(kind, variant, M, N, Kd, 0, 0, 4, 0).name
    ck = K.KernelInfo(kind, variant | 32, M, N, Kd, 0, 0, 4, 0)
    c = ck.config
    again = K.KernelInfo(kind, variant, M, N, Kd, c["block_m"], c["block_n"], 4, c["split_k"])
    assert "ws_kernel" in ck.name and ck.name == again.name and ck.config == again.config
