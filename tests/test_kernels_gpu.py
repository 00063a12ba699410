"""Each HIP kernel alone against a plain PyTorch reference of the same
operation, at sizes other than the engine's, in float32 and in bfloat16."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


def K():
    from lockstep_amd.ops import kernels

    return kernels()


def rel_err(got: torch.Tensor, want: torch.Tensor) -> float:
    got, want = got.double().cpu(), want.double().cpu()
    return float((got - want).abs().max() / want.abs().max().clamp_min(1e-30))


TOL = {torch.float32: 2e-5, torch.bfloat16: 1.5e-2}


# -- matrix product ------------------------------------------------------------

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (1, 1000, 96), (5, 48, 200), (16, 100, 64), (17, 33, 72),
                                   (64, 256, 1024), (65, 130, 260), (37, 3072, 1024), (200, 96, 4100),
                                   (130, 1000, 8), (3, 40, 12),
                                   # tiles of 192 x 128 with rows, columns and K that end inside a tile, and the same
                                   # with K not 16-byte aligned
                                   (2050, 2100, 264), (2050, 2100, 260),
                                   # an odd K: no operand row is 16-byte aligned, in either precision
                                   (200, 90, 101), (9, 50, 37)])
def test_gemm_matches_linear(dtype, m, n, k):
    from lockstep_amd.ops import STORE, STORE_F32, ADD_F32

    g = torch.Generator().manual_seed(m * 1000 + n + k)
    x = torch.randn(m, k, generator=g).to(dtype)
    w = torch.randn(n, k, generator=g).to(dtype)
    want = x.double() @ w.double().T
    xd, wd = x.cuda(), w.cuda()
    out = torch.empty(m, n, dtype=dtype, device="cuda")
    K().gemm(xd, wd, out, STORE)
    assert rel_err(out, want) < TOL[dtype]
    out32 = torch.empty(m, n, dtype=torch.float32, device="cuda")
    K().gemm(xd, wd, out32, STORE_F32)
    assert rel_err(out32, want) < (2e-5 if dtype is torch.float32 else 2e-5 + 0)  # float accumulate: tight in both
    base = torch.randn(m, n, generator=g)
    acc = base.cuda()
    K().gemm(xd, wd, acc, ADD_F32)
    assert rel_err(acc, base.double() + want) < 2e-5


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k,n", [(4096, 4608), (4096, 4613), (4096, 6144), (4096, 6148), (2560, 9210), (2048, 8200), (3584, 2571)])
def test_products_of_few_rows_by_blocks_of_twelve_columns(dtype, k, n):
    """Walks over blocks of 12 columns and, one column block more, of 16 (columns that end inside a block and off a vector, a last round of few
    walkers, one and two groups of rows), against the same rows among 300, which other kernels take: the same bits."""
    from lockstep_amd.ops import ADD_F32, STORE, STORE_F32

    g = torch.Generator().manual_seed(n)
    x = torch.randn(300, k, generator=g).to(dtype).cuda()
    w = torch.randn(n, k, generator=g).to(dtype).cuda()
    start = torch.randn(300, n, generator=g).cuda()
    for epilogue, kind in ((STORE, dtype), (STORE_F32, torch.float32), (ADD_F32, torch.float32)):
        full = start.to(kind, copy=True)
        K().gemm(x, w, full, epilogue)
        for rows in (1, 7, 16, 24, 31, 40, 55):
            part = torch.full((rows + 1, n), 3.0, dtype=kind, device="cuda")
            part[:rows] = start[:rows]
            K().gemm(x[:rows], w, part[:rows], epilogue)
            assert torch.equal(part[:rows], full[:rows]) and (part[rows] == 3.0).all(), (epilogue, rows)


@pytest.mark.parametrize("dtype", DTYPES)
def test_gemm_row_does_not_depend_on_the_batch(dtype):
    """Row i alone, in a 16-row batch, in a 64-row batch and in a 300-row batch:
    same bits (the kernels of few and of many rows share one summation order)."""
    from lockstep_amd.ops import STORE_F32

    g = torch.Generator().manual_seed(7)
    # the last shape has so many columns that 17 to 64 rows already take the ring kernel
    for k, n in ((1024, 272), (3072, 96), (200, 130), (5000, 64), (96, 32768 + 40)):
        x = torch.randn(300, k, generator=g).to(dtype).cuda()
        w = torch.randn(n, k, generator=g).to(dtype).cuda()
        full = torch.empty(300, n, dtype=torch.float32, device="cuda")
        K().gemm(x, w, full, STORE_F32)
        for rows in (1, 16, 17, 64, 65, 128):
            part = torch.empty(rows, n, dtype=torch.float32, device="cuda")
            K().gemm(x[:rows], w, part, STORE_F32)
            assert torch.equal(part, full[:rows]), f"rows={rows} k={k} n={n}"
        for i in (0, 1, 17, 63, 64, 299):
            one = torch.empty(1, n, dtype=torch.float32, device="cuda")
            K().gemm(x[i:i + 1], w, one, STORE_F32)
            assert torch.equal(one[0], full[i]), f"row {i} k={k} n={n}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k,n", [(4096, 4096 + 24), (1000, 16384 + 24), (5120, 4096 + 104), (260, 32768 + 40),
                                 # slices of 512 and some 7,000 columns: tiles of 64 x 64 outputs (float32 64 x 32) from 17 and 32 rows on
                                 (5120, 7168 + 24), (1000, 6144 + 8),
                                 (2048, 8192 + 8), (96, 65536 + 48),
                                 # K of 5,120 over so many columns that tiles of 64 x 128 give every CU one (bfloat16)
                                 (5120, 36864 + 72)])
def test_gemm_with_few_rows_and_many_columns_has_the_same_bits(dtype, k, n):
    """With up to 64 rows and more column blocks than the GPU holds workgroups, a workgroup walks
    several column blocks with its rows of X in registers (the streaming kernel; beyond 32 rows two
    groups of workgroups take 32 rows each).  Every row has the bits it has in a large batch, with
    every epilogue; a row of the sums equals the double precision product."""
    from lockstep_amd.ops import ADD_F32, STORE, STORE_F32

    g = torch.Generator().manual_seed(k + n)
    x = torch.randn(200, k, generator=g).to(dtype).cuda()
    w = (torch.randn(n, k, generator=g) * 0.1).to(dtype).cuda()
    full = torch.empty(200, n, dtype=torch.float32, device="cuda")
    K().gemm(x, w, full, STORE_F32)
    want = x[:3].double().cpu() @ w.double().cpu().T
    assert rel_err(full[:3], want) < 2e-5
    base = torch.randn(64, n, generator=g).cuda()
    for rows in (1, 8, 16, 17, 32, 33, 50, 64):
        part = torch.empty(rows, n, dtype=torch.float32, device="cuda")
        K().gemm(x[:rows], w, part, STORE_F32)
        assert torch.equal(part, full[:rows]), f"rows={rows}"
        stored = torch.empty(rows, n, dtype=dtype, device="cuda")
        K().gemm(x[:rows], w, stored, STORE)
        assert torch.equal(stored, full[:rows].to(dtype)), f"rows={rows}, stored in {dtype}"
        acc = base[:rows].clone()
        K().gemm(x[:rows], w, acc, ADD_F32)
        assert torch.equal(acc, base[:rows] + full[:rows]), f"rows={rows}, added"
    one = torch.empty(1, n, dtype=torch.float32, device="cuda")
    K().gemm(x[31:32], w, one, STORE_F32)
    assert torch.equal(one[0], full[31])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [264, 1088])
def test_gemm_with_many_rows_and_columns_has_the_bits_of_few_rows(dtype, k):
    """2,050 rows by 3,740 columns: 11 x 20 tiles of 192 x 192 outputs fit one round of 256 CUs, so
    bfloat16 takes those (float32 64 x 64 tiles); rows, columns and (with 264) K end inside a tile.
    Every epilogue; rows from all over the product have the bits they have in a product of 40 rows,
    which the skinny kernel computes."""
    from lockstep_amd.ops import ADD_F32, STORE, STORE_F32, SWIGLU, interleave_gate_up

    g = torch.Generator().manual_seed(k)
    m, n = 2050, 3740
    x = torch.randn(m, k, generator=g).to(dtype).cuda()
    w = (torch.randn(n, k, generator=g) * 0.1).to(dtype).cuda()
    full = torch.empty(m, n, dtype=torch.float32, device="cuda")
    K().gemm(x, w, full, STORE_F32)
    want = x[-3:].double().cpu() @ w.double().cpu().T
    assert rel_err(full[-3:], want) < 2e-5
    stored = torch.empty(m, n, dtype=dtype, device="cuda")
    K().gemm(x, w, stored, STORE)
    assert torch.equal(stored, full.to(dtype))
    base = torch.randn(m, n, generator=g).cuda()
    acc = base.clone()
    K().gemm(x, w, acc, ADD_F32)
    assert torch.equal(acc, base + full)
    inter = n // 2
    wi = interleave_gate_up(w[:inter].cpu(), w[inter:].cpu()).cuda()
    gated = torch.empty(m, inter, dtype=dtype, device="cuda")
    K().gemm(x, wi, gated, SWIGLU)
    for first in (0, 100, 1000, 2010):
        rows = slice(first, first + 40)
        part = torch.empty(40, n, dtype=torch.float32, device="cuda")
        K().gemm(x[rows], w, part, STORE_F32)
        assert torch.equal(part, full[rows]), f"rows from {first}"
        part = torch.empty(40, inter, dtype=dtype, device="cuda")
        K().gemm(x[rows], wi, part, SWIGLU)
        assert torch.equal(part, gated[rows]), f"rows from {first}, SwiGLU"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [8, 72, 328, 4424])
@pytest.mark.parametrize("m,n", [(2041, 6152), (2041, 4091), (1501, 6139), (1003, 6139), (1501, 4088), (1003, 4096), (1003, 2044),
                                 (64, 32700), (300, 1000), (65, 16), (130, 3)])
def test_every_tile_of_the_products_has_the_bits_of_few_rows(dtype, k, m, n):
    """Sizes over the tiles of the ring kernel (bfloat16: all but 256 x 192 with a plain epilogue, see the test of every tile by
    name; float32: 64 x 64), with rows and columns that end inside a tile, K of less than a stage, K that ends inside a stage and inside a slice, and columns that no vector store fits:
    five rows at a time, which the kernels of a wave a slice compute, have the same bits."""
    from lockstep_amd.ops import ADD_F32, STORE, STORE_F32, SWIGLU

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
    x[-1], w[-1] = float("inf"), float("nan")               # a row and a column must not reach another one
    full = torch.full((m, n), 7.0, device="cuda")
    K().gemm(x, w, full, STORE_F32)
    stored = torch.empty(m, n, dtype=dtype, device="cuda")
    K().gemm(x, w, stored, STORE)
    assert torch.equal(stored[:-1, :-1], full[:-1, :-1].to(dtype))
    base = torch.randn(m, n, generator=g, device="cuda")
    acc = base.clone()
    K().gemm(x, w, acc, ADD_F32)
    assert torch.equal(acc[:-1, :-1], base[:-1, :-1] + full[:-1, :-1])
    gated = None
    if n % 32 == 8:                                          # as interleaved gate and up rows
        n_gated = n - 8
        gated = torch.empty(m, n_gated // 2, dtype=dtype, device="cuda")
        K().gemm(x, w[:n_gated].contiguous(), gated, SWIGLU)
    want = x[:2].double() @ w[:-1].double().T
    assert rel_err(full[:2, :-1], want) < 2e-5
    for first in sorted({0, m // 2, m - 7}):
        rows = slice(first, first + 5)
        part = torch.empty(5, n, device="cuda")
        K().gemm(x[rows], w, part, STORE_F32)
        assert torch.equal(part[:, :-1], full[rows, :-1]), f"rows from {first}"
        assert torch.isnan(full[rows, -1]).all()
        if gated is not None:
            part = torch.empty(5, n_gated // 2, dtype=dtype, device="cuda")
            K().gemm(x[rows], w[:n_gated].contiguous(), part, SWIGLU)
            assert torch.equal(part, gated[rows]), f"rows from {first}, SwiGLU"


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_of_x_further_apart_than_offsets_of_32_bits_reach(dtype):
    """64 rows of X that span 4 GiB and more (a view into a wide buffer): the product and its slice sums have the bits of the
    same rows side by side."""
    from lockstep_amd.ops import STORE_F32

    size = torch.finfo(dtype).bits // 8
    ldx, k = (1 << 26) // size + 16, 1024
    g = torch.Generator(device="cuda").manual_seed(size)
    near = torch.randn(65, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(4096, k, generator=g, device="cuda") * 0.1).to(dtype)
    far = torch.empty(64 * ldx + k, dtype=dtype, device="cuda").as_strided((65, k), (ldx, 1))
    far.copy_(near)
    out, want = (torch.empty(65, 4096, device="cuda") for _ in range(2))
    K().gemm(far, w, out, STORE_F32)
    K().gemm(near, w, want, STORE_F32)
    assert torch.equal(out, want)
    sums, expected = (torch.empty(K().gemm_slices_count(k), 64, 4096, device="cuda") for _ in range(2))
    K().gemm_slices(far[:64], w, sums)
    K().gemm_slices(near[:64], w, expected)
    assert torch.equal(sums, expected)
    del far
    torch.cuda.empty_cache()


@pytest.mark.parametrize("big", ["weights", "rows"])
def test_what_a_stage_reads_behind_the_last_column_of_an_operand_of_4_gib(big):
    """An operand that goes on for more than 4 GiB behind the first tile, K that ends inside a stage: the last stage's loads behind K
    read zeros and not the operand, whatever its bytes are a byte off.  The first and the last tile have the bits of the same rows alone."""
    from lockstep_amd.ops import STORE_F32

    k, many, few = 4104, 530_000, 97                             # 4.05 GiB
    g = torch.Generator(device="cuda").manual_seed(k)
    large = torch.empty(many, k, dtype=torch.bfloat16, device="cuda").normal_(0, 0.1, generator=g)
    small = torch.randn(few, k, generator=g, device="cuda").to(torch.bfloat16)
    x, w = (small, large) if big == "weights" else (large, small)
    out = torch.empty(x.shape[0], w.shape[0], device="cuda")
    K().gemm(x, w, out, STORE_F32)
    for part in (slice(0, 300), slice(many - 300, many)):
        a, b = (x, w[part]) if big == "weights" else (x[part], w)
        want = torch.empty(a.shape[0], b.shape[0], device="cuda")
        K().gemm(a, b, want, STORE_F32)
        assert torch.equal(out[:, part] if big == "weights" else out[part], want)
        exact = a[:4].double() @ b.double().T
        assert rel_err(want[:4], exact) < 2e-5
    del large, x, w, out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,k", [(40, 8), (100, 264), (1000, 1032), (4099, 2056), (6148, 4096), (9000, 4424)])
def test_few_rows_read_by_whole_pieces_have_the_bits_of_element_by_element_reads(dtype, n, k):
    """Rows of X one element behind a 16-byte boundary take the general loads, aligned ones buffer loads: columns that end inside a
    block, slices that end inside a round of loads, walks of an even and an odd number of blocks; the slice sums likewise."""
    from lockstep_amd.ops import STORE_F32

    g = torch.Generator(device="cuda").manual_seed(n + k)
    x = torch.randn(64, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
    off = torch.empty(64 * k + 8, dtype=dtype, device="cuda")[1:1 + 64 * k].view(64, k)
    off.copy_(x)
    for m in (1, 3, 16, 17, 40, 64):
        a, b = (torch.full((m, n), float("nan"), device="cuda") for _ in range(2))
        K().gemm(x[:m], w, a, STORE_F32)
        K().gemm(off[:m], w, b, STORE_F32)
        assert torch.equal(a, b), m
        a, b = (torch.full((K().gemm_slices_count(k), m, n), float("nan"), device="cuda") for _ in range(2))
        K().gemm_slices(x[:m], w, a)
        K().gemm_slices(off[:m], w, b)
        assert torch.equal(a, b), f"slice sums, {m}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k,n", [(2048, 9000), (4096, 8209)])
def test_walks_over_aligned_rows_too_far_apart_for_whole_pieces(dtype, k, n):
    """Three rows of X whose distance puts 65 of them past 2 GiB: the streaming kernel's general instance, whose walks end at
    different blocks, with the bits of the rows side by side."""
    from lockstep_amd.ops import STORE_F32

    size = torch.finfo(dtype).bits // 8
    ldx = (1 << 25) // size + 16
    g = torch.Generator(device="cuda").manual_seed(size + k)
    near = torch.randn(3, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
    far = torch.empty(2 * ldx + k, dtype=dtype, device="cuda").as_strided((3, k), (ldx, 1))
    far.copy_(near)
    out, want = (torch.empty(3, n, device="cuda") for _ in range(2))
    K().gemm(far, w, out, STORE_F32)
    K().gemm(near, w, want, STORE_F32)
    assert torch.equal(out, want)


# (rows, columns) that take each tile of the ring kernel, in the order of RingTile, with both ending inside a tile
RING_TILE_SIZES = [(2041, 4448), (1003, 6176), (1501, 5408), (1003, 5408), (700, 5408), (500, 4128), (130, 5472), (300, 5472), (65, 5536),
                   (97, 4064), (97, 96)]


@pytest.mark.parametrize("k", [72, 328])
@pytest.mark.parametrize("m,n", RING_TILE_SIZES)
def test_every_ring_tile_with_every_epilogue_has_the_bits_of_few_rows(m, n, k):
    """Each tile by the name that the dispatch gives it, K that ends inside the second stage and inside a slice."""
    from lockstep_amd.ops import ADD_F32, STORE, STORE_F32, SWIGLU

    dtype = torch.bfloat16
    tile = RING_TILE_SIZES.index((m, n))
    assert [K().gemm_ring_tile(dtype, e, m, n, k) for e in (STORE, STORE_F32, ADD_F32, SWIGLU)] == [tile] * 4
    assert [K().gemm_ring_tile(dtype, e, 5, n, k) for e in (STORE, STORE_F32, ADD_F32, SWIGLU)] == [-1] * 4
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
    base = torch.randn(m, n, generator=g, device="cuda")
    act = torch.tensor([0.8, 0.3], device="cuda")

    def run(epilogue, rows):
        out = (base[rows].clone() if epilogue == ADD_F32 else
               torch.empty(rows.stop - rows.start, n // 2 if epilogue == SWIGLU else n, device="cuda",
                           dtype=torch.float32 if epilogue == STORE_F32 else dtype))
        if epilogue == "xielu":
            K().gemm_xielu(x[rows], w, out, act)
        else:
            K().gemm(x[rows], w, out, epilogue)
        return out

    for epilogue in (STORE, STORE_F32, ADD_F32, SWIGLU, "xielu"):
        full = run(epilogue, slice(0, m))
        for first in (0, m // 2, m - 5):
            rows = slice(first, first + 5)
            assert torch.equal(run(epilogue, rows), full[rows]), (epilogue, first)


# (rows, columns, K, whether SwiGLU) on both sides of the lines between the ring kernel and the others and of those between its tiles, and the
# tile it takes (8, 9, 10: 64 x 64, 32 x 64, 32 x 32)
RING_LINES = {
    torch.float32: [(8, 12288, 512, False, -1), (9, 4112, 256, False, 10), (9, 4112, 252, False, -1), (9, 4096, 512, False, -1), (17, 4093, 384, False, 10),
                    (17, 4093, 388, False, -1), (17, 4112, 512, False, 10), (32, 4096, 516, False, -1), (33, 4093, 516, False, 10), (33, 24, 8, False, 10),
                    (64, 16384, 512, False, 8), (64, 16401, 512, False, 10), (130, 16381, 72, False, 8), (97, 12289, 72, False, 8), (16, 8192, 512, True, 10),
                    (16, 8192, 516, True, -1), (8, 8224, 520, True, 10), (8, 29984, 520, True, 10), (8, 30016, 520, True, -1), (9, 30016, 520, True, 10),
                    (17, 8192, 520, True, 10), (33, 24544, 72, True, 8)],
    torch.bfloat16: [(16, 4096, 1032, False, -1), (16, 4109, 384, False, 10), (16, 4109, 320, False, -1), (16, 4109, 648, False, 10), (16, 4109, 632, False, -1), (8, 4109, 640, False, 10),
                     (8, 4109, 632, False, -1), (8, 16381, 640, False, 9), (8, 16400, 640, False, -1), (8, 16400, 2048, False, 10),
                     (8, 24608, 2048, False, -1), (7, 32768, 128, False, 9), (7, 32752, 128, False, -1), (8, 32768, 320, False, 9),
                     (8, 32768, 312, False, -1), (7, 32768, 320, False, -1), (9, 32768, 136, False, 9), (7, 65473, 72, False, 7),
                     (17, 4093, 320, False, 10), (17, 4093, 328, False, -1), (32, 4091, 4104, False, 10), (32, 4096, 4088, False, -1), (24, 4096, 4104, False, -1),
                     (17, 4112, 264, False, 10), (17, 4112, 248, False, -1), (17, 20000, 248, False, 7), (33, 24, 8, False, 10),
                     (33, 4097, 72, False, 9), (64, 8192, 264, False, 9), (64, 8193, 264, False, 8), (64, 8193, 2048, False, 8),
                     (97, 4091, 72, False, 9), (97, 4097, 72, False, 8), (257, 909, 4424, False, 9), (32, 16384, 520, False, 9),
                     (32, 16416, 520, False, 7), (32, 24544, 512, False, 9), (32, 24544, 520, False, 7), (31, 24544, 2056, True, 10),
                     (31, 24608, 2056, True, 7), (33, 24544, 2056, True, 7), (8, 4096, 640, True, 10), (8, 4096, 576, True, -1),
                     (9, 4096, 320, True, 10), (9, 4096, 256, True, -1), (16, 8192, 328, True, -1), (16, 8192, 2600, True, 10),
                     (16, 8192, 2584, True, -1), (16, 8224, 328, True, 9), (17, 96, 8, True, 10), (1, 6144, 1024, True, 10)],
}


@pytest.mark.parametrize("dtype", DTYPES)
def test_products_on_both_sides_of_the_lines_of_the_ring_kernel_have_the_same_bits(dtype):
    """Weights one element behind a 16-byte boundary go to kernels of another kind (a wave a slice, tiles through registers): the
    same bits.  The sum of every element is at most sum(|x||w|) 2^-24 (K + K / 256) off (each addition rounds once)."""
    from lockstep_amd.ops import ADD_F32, STORE_F32, SWIGLU

    for m, n, k, gated, tile in RING_LINES[dtype]:
        epilogue = SWIGLU if gated else STORE_F32
        assert K().gemm_ring_tile(dtype, epilogue, m, n, k) == tile, (m, n, k, gated)
        g = torch.Generator(device="cuda").manual_seed(m + n + k)
        x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
        w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
        sound = max(1, m - 1)                                    # rows without an infinity: a row must not reach another one
        x[sound:] = float("inf")
        off = torch.empty(n * k + 8, dtype=dtype, device="cuda")[1:1 + n * k].view(n, k)
        off.copy_(w)
        a, b = (torch.full((m, n // 2 if gated else n), 7.0, dtype=dtype if gated else torch.float32, device="cuda") for _ in range(2))
        K().gemm(x, w, a, epilogue)
        K().gemm(x, off, b, epilogue)
        assert torch.equal(a[:sound], b[:sound]), (m, n, k, gated)
        if not gated:
            want, most = x[:sound].double() @ w.double().T, x[:sound].double().abs() @ w.double().abs().T
            assert ((a[:sound] - want).abs() <= most * 2.0 ** -24 * (k + k / 256 + 1)).all(), (m, n, k)
            K().gemm(x, w, a, ADD_F32)
            assert torch.equal(a[:sound], b[:sound] + b[:sound]), (m, n, k)


# (rows, columns, K) of slice sums, and (rows of the tile, slices a workgroup) of the ring kernel that computes them in bfloat16 and in float32
SLICES_PLANS = [(3, 4096, 4096, (0, 0), (0, 0)), (4, 4096, 4096, (32, 4), (0, 0)), (17, 1028, 1288, (0, 0), (0, 0)), (33, 1024, 8, (0, 0), (0, 0)),
                (40, 260, 328, (0, 0), (0, 0)), (65, 508, 2048, (32, 1), (0, 0)), (32, 1020, 4424, (32, 1), (0, 0)), (64, 1024, 2048, (32, 1), (0, 0)),
                (8, 5116, 8192, (32, 2), (0, 0)), (24, 8188, 1032, (32, 4), (0, 0)), (64, 4092, 1032, (64, 1), (64, 1)),
                (64, 1020, 3072, (64, 1), (64, 1)), (128, 5116, 5120, (64, 1), (64, 1)), (56, 8188, 4424, (64, 1), (64, 1)),
                (33, 4092, 4096, (64, 2), (64, 2)), (64, 4092, 4096, (64, 2), (64, 2)), (200, 1024, 3072, (64, 2), (64, 1)),
                (256, 4096, 520, (64, 2), (64, 1)), (33, 12284, 3080, (64, 4), (64, 1)),
                (8, 4092, 12288, (32, 2), (0, 0)), (6, 1468, 9576, (32, 2), (0, 0)), (18, 2236, 14336, (32, 1), (0, 0)), (32, 1020, 9576, (32, 1), (0, 0)),
                (24, 3004, 9576, (32, 1), (0, 0)), (6, 6656, 2304, (0, 0), (0, 0)), (10, 6784, 1128, (0, 0), (0, 0)), (17, 1404, 3072, (32, 2), (0, 0)),
                (17, 1404, 3080, (0, 0), (0, 0)), (8, 4096, 2560, (0, 0), (0, 0)), (256, 512, 512, (0, 0), (0, 0))]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k,plan,plan_f32", SLICES_PLANS)
def test_slice_sums_by_either_tile_add_up_to_the_product(dtype, m, n, k, plan, plan_f32):
    """Slice sums of every plan, with rows and columns that end inside a tile and a last workgroup with fewer slices: every sum is there, they
    have the bits that another kernel gives for weights off a 16-byte boundary, and added in ascending order they are the product, bit for bit."""
    from lockstep_amd.ops import STORE_F32

    if m > K().gemm_slices_max_rows(k, dtype):
        pytest.skip("more rows than the slice sums take")
    assert K().gemm_slices_plan(dtype, m, n, k) == (plan if dtype is torch.bfloat16 else plan_f32)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
    off = torch.empty(n * k + 8, dtype=dtype, device="cuda")[1:1 + n * k].view(n, k)
    off.copy_(w)
    sums, others = (torch.full((K().gemm_slices_count(k), m, n), float("nan"), device="cuda") for _ in range(2))
    K().gemm_slices(x, w, sums)
    K().gemm_slices(x, off, others)
    assert torch.equal(sums, others)
    want = torch.empty(m, n, device="cuda")
    K().gemm(x, w, want, STORE_F32)
    total = torch.zeros(m, n, device="cuda")
    for part in sums:
        total = total + part
    assert torch.equal(total, want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,k,gated", [(16352, 200, False), (16352, 200, True), (32768 + 40, 96, False), (32768, 72, True)])
def test_products_off_a_16_byte_boundary_with_few_rows_have_the_bits_of_aligned_ones(dtype, n, k, gated):
    """Weights one element behind a 16-byte boundary: 17 to 64 rows over so many columns go to tiles, fewer to a wave a slice."""
    from lockstep_amd.ops import STORE_F32, SWIGLU

    g = torch.Generator(device="cuda").manual_seed(n + k)
    x = torch.randn(64, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).to(dtype)
    off = torch.empty(n * k + 8, dtype=dtype, device="cuda")[1:1 + n * k].view(n, k)
    off.copy_(w)
    for m in (5, 16, 17, 32, 33, 64):
        a, b = (torch.empty(m, n // 2 if gated else n, dtype=dtype if gated else torch.float32, device="cuda") for _ in range(2))
        K().gemm(x[:m], w, a, SWIGLU if gated else STORE_F32)
        K().gemm(x[:m], off, b, SWIGLU if gated else STORE_F32)
        assert torch.equal(a, b), m


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inter,k", [(4096 + 40, 4096), (16384 + 72, 1024), (25600, 5120)])
def test_swiglu_with_few_rows_and_many_columns_has_the_same_bits(dtype, inter, k):
    from lockstep_amd.ops import SWIGLU, interleave_gate_up

    g = torch.Generator().manual_seed(inter + k)
    x = torch.randn(150, k, generator=g).to(dtype).cuda()
    gate = (torch.randn(inter, k, generator=g) * 0.05).to(dtype)
    up = (torch.randn(inter, k, generator=g) * 0.05).to(dtype)
    w = interleave_gate_up(gate, up).cuda()
    full = torch.empty(150, inter, dtype=dtype, device="cuda")
    K().gemm(x, w, full, SWIGLU)
    want = torch.nn.functional.silu(x[:2].double().cpu() @ gate.double().T) * (x[:2].double().cpu() @ up.double().T)
    assert rel_err(full[:2], want) < TOL[dtype]
    for rows in (1, 8, 16, 20, 32, 40, 64):
        part = torch.empty(rows, inter, dtype=dtype, device="cuda")
        K().gemm(x[:rows], w, part, SWIGLU)
        assert torch.equal(part, full[:rows]), f"rows={rows}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [1024, 4096, 5120])
def test_the_full_vocabulary_head_against_double_precision(dtype, k):
    """151,936 columns (the streaming kernel for few rows, tiles of 64 rows up to 64 rows, larger ones
    beyond) at 1, 8, 64 and 200 rows: every row equals the double-precision product and has the
    same bits at every number of rows."""
    from lockstep_amd.ops import STORE_F32

    vocab = 151936
    g = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn(200, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(vocab, k, generator=g, device="cuda") * 0.05).to(dtype)
    want = torch.cat([x.double() @ w[lo:lo + 16384].double().T for lo in range(0, vocab, 16384)], dim=1)
    full = None
    for rows in (200, 1, 8, 64):
        out = torch.full((rows, vocab), float("nan"), device="cuda")
        K().gemm(x[:rows], w, out, STORE_F32)
        assert rel_err(out, want[:rows]) < 2e-5, rows
        if full is None:
            full = out
        assert torch.equal(out, full[:rows]), rows
    del w, want, full
    torch.cuda.empty_cache()


@pytest.mark.parametrize("vocab", [7, 1000, 4099, 151936])
def test_the_sampling_kernel_picks_the_host_samplers_token(vocab):
    """Temperature and nucleus sampling on the device against the host procedure (float64, sorted): the same
    token for every row, with spread-out and with quantised logits (many equal values: the order among
    equals is the order of the ids), small and large nuclei, several temperatures; twice the same."""
    from lockstep_amd.sampling import philox
    from lockstep_amd.sampling.sampler import top_p as host_top_p

    n = 48 if vocab < 100000 else 12
    g = torch.Generator().manual_seed(vocab)
    logits = torch.randn(n + 3, vocab, generator=g) * (0.5 + 3 * torch.rand(n + 3, 1, generator=g))
    logits[::5] = torch.round(logits[::5] * 2) / 2
    logits[1, : vocab // 2] = logits[1, 0]                          # half of the row is one value
    rows = torch.randperm(n + 3, generator=g)[:n].to(torch.int32)
    temperature = [[0.3, 0.8, 1.0, 1.7][i % 4] for i in range(n)]
    nucleus = [[1.0, 0.9, 0.5, 0.05, 0.999, 0.0][i % 6] for i in range(n)]
    seed = 7 + (1 << 40)                          # both halves of the key in use
    # the host procedure with the same seed, uid and position (positions beyond 32 bits too)
    positions = [i if i % 7 else (5 << 32) + i for i in range(n)]
    want = [host_top_p(logits[int(rows[i])], seed, "kernel", positions[i], nucleus[i], temperature[i]) for i in range(n)]
    dev = logits.cuda()
    requests = [(int(rows[i]), temperature[i], nucleus[i], seed ^ philox.uid_key("kernel"), positions[i]) for i in range(n)]
    out = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    K().sample_top_p(dev, requests, out)
    assert out.cpu().tolist() == want
    again = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    K().sample_top_p(dev, requests, again)
    assert torch.equal(out, again)
    assert len(set(want)) > 1


def sample_among(kernels, dev, requests, n_rows: int, order_seed: int):
    """The tokens of ``requests`` when they are sampled in one call of ``n_rows`` rows (the others
    being further draws from the same logits rows), in a shuffled order."""
    base = len(requests)
    extra = [(i % base, 0.5 + (i % 7) / 4, [1.0, 0.8][i % 2], 900 + i, 50000 + i) for i in range(max(0, n_rows - base))]
    every = list(requests[:n_rows]) + extra
    order = torch.randperm(len(every), generator=torch.Generator().manual_seed(order_seed)).tolist()
    out = torch.full((len(every),), -1, dtype=torch.int32, device="cuda")
    kernels.sample_top_p(dev, [every[j] for j in order], out)
    picked = out.cpu().tolist()
    tokens = [None] * len(every)
    for place, j in enumerate(order):
        tokens[j] = picked[place]
    return tokens[:min(n_rows, base)]


@pytest.mark.parametrize("vocab", [1000, 151936])
def test_a_sampled_row_gets_the_same_token_beside_any_number_of_other_rows(vocab):
    """The same logits rows sampled alone and in calls of 24, 33, 64 and 200 rows: the same tokens.
    Half of the rows are spread-out logits with random nuclei; the other half are made so that a
    change in the order of any sum would show (``sampling_rows_on_boundaries``: the positive
    control of this test runs them against a sampler whose cut depends on the rows of the call)."""
    from helpers import sampling_rows_on_boundaries
    from lockstep_amd.sampling import philox

    g = torch.Generator().manual_seed(vocab + 1)
    spread = torch.randn(12, vocab, generator=g) * 2.0
    spread[::2] = torch.round(spread[::2] * 4) / 4
    spread[3, : vocab // 3] = 1.25
    spread[5] = 0.0                                                 # one value only: the draw counts ties off
    sharp, on_boundaries = sampling_rows_on_boundaries(vocab, rows=12)
    dev = torch.cat([spread, sharp]).cuda()
    key = philox.uid_key("same-row")
    requests = [(i, [0.7, 1.0, 1.9][i % 3], [1.0, 0.9, 0.3, 0.999][i % 4], (11 + i) ^ key, 1000 + 17 * i) for i in range(12)]
    requests += [(12 + row, t, p, k, pos) for row, t, p, k, pos in on_boundaries]
    alone = []
    for request in requests:                                        # every request in a call of its own
        out = torch.full((1,), -1, dtype=torch.int32, device="cuda")
        K().sample_top_p(dev, [request], out)
        alone.append(int(out.item()))
    assert all(0 <= t < vocab for t in alone)
    for n_rows in (len(requests), 33, 64, 200):
        assert sample_among(K(), dev, requests, n_rows, n_rows) == alone, f"{n_rows} rows in the call"


def test_the_sampler_takes_greedy_and_drawn_rows_of_one_step_together():
    from lockstep_amd.sampling import Sampler
    from lockstep_amd.sampling.sampler import top_p as host_top_p

    class Row:
        def __init__(self, uid, seed, temperature, nucleus, total):
            self.uid, self.seed, self.temperature, self.top_p, self._total = uid, seed, temperature, nucleus, total

        def total_tokens(self):
            return self._total

    g = torch.Generator().manual_seed(3)
    logits = torch.randn(6, 5003, generator=g) * 2
    requests = [Row("a", 1, 0.0, 1.0, 5), Row("b", 2, 0.7, 0.9, 9), Row("c", 3, 0.0, 1.0, 2), Row("d", 4, 1.3, 1.0, 40),
                Row("e", 5, 0.2, 0.3, 7), Row("f", 6, 1.0, 0.95, 1)]
    want = [host_top_p(logits[i], r.seed, r.uid, r.total_tokens() - 1, r.top_p, r.temperature) for i, r in enumerate(requests)]
    assert Sampler(K()).sample(logits.cuda(), requests) == want


def test_gemm_refuses_mismatched_operands():
    from lockstep_amd.ops import KernelError

    x = torch.zeros(4, 32, device="cuda")
    w = torch.zeros(8, 48, device="cuda")
    with pytest.raises(KernelError):
        K().gemm(x, w, torch.zeros(4, 8, device="cuda"))


@pytest.mark.parametrize("out_dtype", DTYPES)
@pytest.mark.parametrize("activation", ["none", "silu", "gelu_tanh", "gelu", "relu"])
@pytest.mark.parametrize("rows,width", [(1, 40), (7, 1000), (70, 3072)])
def test_bias_and_activation_pass_against_torch(out_dtype, activation, rows, width):
    """``act(x + bias)`` and its gated form ``act(gate + b) * (up + b)``, with and without a bias, also in place."""
    g = torch.Generator().manual_seed(rows + width)
    acts = {"none": lambda v: v, "silu": torch.nn.functional.silu, "relu": torch.relu,
            "gelu": torch.nn.functional.gelu, "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}
    tol = 2e-6 if out_dtype is torch.float32 else 5e-3
    for gated in (False, True):
        x = torch.randn(rows, width * (2 if gated else 1) + 8, generator=g).cuda()[:, : width * (2 if gated else 1)]
        for bias in (None, torch.randn(x.shape[1], generator=g).cuda()):
            out = torch.full((rows, width), float("nan"), dtype=out_dtype, device="cuda")
            K().bias_act(x, bias, out, activation, gated=gated)
            v = x.double() + (bias.double() if bias is not None else 0.0)
            want = acts[activation](v[:, :width]) * (v[:, width:] if gated else 1.0)
            assert rel_err(out, want) < tol, (activation, gated, bias is not None)
    x = torch.randn(rows, width, generator=g).cuda()
    bias = torch.randn(width, generator=g).cuda()
    want = acts[activation](x.double() + bias.double())
    K().bias_act(x, bias, x, activation)                        # in place
    assert rel_err(x, want) < 2e-6
    from lockstep_amd.ops import KernelError
    with pytest.raises(KernelError, match="not built"):
        K().bias_act(x, None, x, "swish7")
    with pytest.raises(KernelError, match="float32 \\["):
        K().bias_act(x, None, torch.empty(rows, width + 1, device="cuda"), "none")


# -- norm --------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,width,eps", [(1, 64, 1e-6), (7, 96, 1e-5), (48, 1024, 1e-6), (3, 5120, 1e-6),
                                            (5, 100, 1e-3)])
def test_rmsnorm_matches_formula(dtype, rows, width, eps):
    g = torch.Generator().manual_seed(width)
    x = torch.randn(rows, width, generator=g) * 3
    w = 1 + 0.1 * torch.randn(width, generator=g)
    want = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + eps) * w.double()
    out = torch.empty(rows, width, dtype=dtype, device="cuda")
    K().rmsnorm(x.cuda(), w.cuda(), out, eps)
    assert rel_err(out, want) < (1e-6 if dtype is torch.float32 else 5e-3)
    lib = torch.nn.functional.rms_norm(x, (width,), w, eps)
    assert rel_err(out, lib) < (1e-6 if dtype is torch.float32 else 5e-3)
    # selected rows, and a row alone gives the same bits as in the batch
    idx = torch.tensor([rows - 1, 0], dtype=torch.int32, device="cuda")
    sel = torch.empty(2, width, dtype=dtype, device="cuda")
    K().rmsnorm(x.cuda(), w.cuda(), sel, eps, idx)
    assert torch.equal(sel[0], out[rows - 1]) and torch.equal(sel[1], out[0])


# -- SwiGLU, embedding, arg-max --------------------------------------------------------

@pytest.mark.parametrize("dtype", DTYPES)
def test_swiglu_matches_silu_times_up(dtype):
    g = torch.Generator().manual_seed(1)
    gu = (torch.randn(7, 2 * 300, generator=g) * 2).to(dtype)
    want = torch.nn.functional.silu(gu[:, :300].double()) * gu[:, 300:].double()
    out = torch.empty(7, 300, dtype=dtype, device="cuda")
    K().swiglu(gu.cuda(), out)
    assert rel_err(out, want) < (1e-6 if dtype is torch.float32 else 5e-3)
    zero = torch.zeros(2, 64, dtype=dtype, device="cuda")
    out0 = torch.ones(2, 32, dtype=dtype, device="cuda")
    K().swiglu(zero, out0)
    assert torch.count_nonzero(out0) == 0


@pytest.mark.parametrize("dtype", DTYPES)
def test_embedding_gathers_rows(dtype):
    table = torch.randn(1000, 96).to(dtype)
    ids = torch.tensor([0, 999, 5, 5, 731], dtype=torch.int32)
    out = torch.empty(5, 96, dtype=torch.float32, device="cuda")
    K().embed(ids.cuda(), table.cuda(), out)
    assert torch.equal(out.cpu(), table[ids.long()].float())


def test_argmax_takes_the_lowest_index_among_maxima():
    x = torch.randn(6, 151936)
    x[1, 77] = x[1, 150000] = 50.0
    x[2, :] = 1.0
    x[3, 151935] = 60.0
    out = torch.empty(6, dtype=torch.int32, device="cuda")
    K().argmax(x.cuda(), out)
    want = [int(torch.nonzero(r == r.max())[0]) for r in x]
    assert out.cpu().tolist() == want
    assert want[1] == 77 and want[2] == 0 and want[3] == 151935


def test_argmax_with_more_rows_than_the_static_scratch_holds():
    """Beyond 16,384 (row, chunk) pairs the wrapper brings a scratch buffer, and a larger call
    after a smaller one grows it; the results are those of the static path."""
    k = K()
    g = torch.Generator().manual_seed(5)
    for rows in (2100, 2900):                       # 3 chunks a row: 6,300 and 8,700 pairs, the static array
        x = torch.randn(rows, 9000, generator=g)
        x[:, 8999] = x.max(dim=1).values            # a tie with the last column: the lower index wins
        out = torch.empty(rows, dtype=torch.int32, device="cuda")
        k.argmax(x.cuda(), out)
        assert torch.equal(out.long().cpu(), (x == x.max(1, keepdim=True).values).int().argmax(1))
    for rows in (5600, 7000):                       # 16,800 and 21,000 pairs: beyond the static array, growing
        assert rows * 3 > k.ARGMAX_STATIC_PAIRS
        x = torch.randn(rows, 9000, generator=g)
        out = torch.empty(rows, dtype=torch.int32, device="cuda")
        k.argmax(x.cuda(), out)
        assert torch.equal(out.long().cpu(), x.argmax(dim=1))
    small = torch.tensor([[1.0, 5.0, 5.0, 5.0, 2.0]]).cuda()
    one = torch.empty(1, dtype=torch.int32, device="cuda")
    K().argmax(small, one)
    assert one.item() == 1
    # widths and row strides that are no multiple of four, maxima at the edges of a chunk, NaN, a view
    g = torch.Generator().manual_seed(3)
    for width in (4095, 4096, 4097, 8191, 12289, 50001):
        y = torch.randn(5, width + 3, generator=g)
        y[0, min(4095, width - 1)] = 9.0
        y[1, min(4096, width - 1)] = 9.0
        y[2, width - 1] = 9.0
        y[3, 0] = float("nan")
        y[4, :] = float("nan")
        view = y.cuda()[:, :width]
        got = torch.empty(5, dtype=torch.int32, device="cuda")
        K().argmax(view, got)
        ref = y[:, :width].clone()
        ref[ref != ref] = float("-inf")
        want = [int(torch.nonzero(r == r.max())[0]) for r in ref]
        want[4] = 0
        assert got.cpu().tolist() == want, width


# -- norm + rotation + cache write, attention ---------------------------------------------

def naive_attention(q, k, v, q_start, scale, window=None):
    """q [Tq,nq,d], k,v [Tk,nkv,d] in float64; explicit max-subtract softmax."""
    tq, nq, d = q.shape
    tk, nkv, _ = k.shape
    g = nq // nkv
    k = k.repeat_interleave(g, dim=1)
    v = v.repeat_interleave(g, dim=1)
    s = torch.einsum("qhd,khd->hqk", q, k) * scale
    qp = torch.arange(q_start, q_start + tq)[:, None]
    kp = torch.arange(tk)[None, :]
    hidden = kp > qp
    if window:
        hidden = hidden | (qp - kp >= window)
    s = s.masked_fill(hidden[None], float("-inf"))
    m = s.max(-1, keepdim=True).values
    e = (s - m).exp()
    return torch.einsum("hqk,khd->qhd", e / e.sum(-1, keepdim=True), v)


class PagedCase:
    """Lay keys and values into pages through the engine's own write kernel."""

    def __init__(self, dtype, nq, nkv, d, page_size, n_tokens, shuffle_seed=None, extra_pages=3):
        self.dtype, self.nq, self.nkv, self.d, self.ps = dtype, nq, nkv, d, page_size
        n_pages = -(-n_tokens // page_size)
        order = list(range(n_pages + extra_pages))
        if shuffle_seed is not None:
            g = torch.Generator().manual_seed(shuffle_seed)
            order = torch.randperm(n_pages + extra_pages, generator=g).tolist()
        self.table = torch.full((2, n_pages + 1), -1, dtype=torch.int32)
        self.table[1, :n_pages] = torch.tensor(order[:n_pages], dtype=torch.int32)
        self.table = self.table.cuda()
        total = n_pages + extra_pages
        self.k_pages = torch.full((total, nkv, page_size, d), float("nan"), dtype=dtype, device="cuda")
        self.v_pages = torch.full((total, nkv, d, page_size), float("nan"), dtype=dtype, device="cuda")

    def seqs(self, q_start, q_len):
        return torch.tensor([0, q_len, q_start, q_start + q_len, 1, 0, 0, 0], dtype=torch.int32).cuda()

    def write(self, qkv, q_start, q_norm=None, k_norm=None, eps=1e-6, cos=None, sin=None, rot=0):
        t = qkv.shape[0]
        tok_seq = torch.zeros(t, dtype=torch.int32, device="cuda")
        tok_pos = torch.arange(q_start, q_start + t, dtype=torch.int32, device="cuda")
        K().qk_rope_kv(qkv, t, self.nq, self.nkv, self.d, q_norm, k_norm, eps, cos, sin, rot, tok_seq, tok_pos,
                       self.seqs(q_start, t), q_start + t - 1, self.table, self.k_pages, self.v_pages, self.ps, True)

    def attend(self, qkv, q_start, scale, window=0, force_split=None, variant=0, repeat=1, span=1, pad_splits=0,
               few_rows=False):
        """``few_rows``: tell the fold that no request has more than 16 rows (it then takes the kernel that
        asks for many splits at a time).  ``span``: splits one work item walks when the request is cut (the cooperative kernel takes more
        than one and leaves a partial result for each); ``pad_splits``: lay the items out for that many
        more splits than the request has (as the fixed-shape lists of graph-replayed steps do)."""
        from lockstep_amd.ops import kernels

        t = qkv.shape[0]
        tile, split = kernels().attention_geometry(self.d)
        g = self.nq // self.nkv
        rows = t * g
        kv_len = q_start + t
        lo = max(0, q_start - window + 1) if window else 0
        split_lo = lo // split
        n_splits = (kv_len - 1) // split + 1 - split_lo
        use_split = (rows <= 64 and n_splits > 1) if force_split is None else force_split
        items, combine, part_rows = [], [], 0
        br = kernels().attention_block_rows(self.d, variant)       # rows of a work item's row block
        if use_split:
            n_splits += pad_splits
            part_rows = self.nkv * rows * n_splits
            for b in range(-(-rows // br)):
                for s in range(split_lo, split_lo + n_splits, span):
                    items += [0, b, s, min(s + span, split_lo + n_splits), 0, n_splits, split_lo, 0]
            for b in range(-(-rows // 64)):
                combine += [0, b, 0, n_splits]
        else:
            for b in range(-(-rows // br)):
                first = q_start + (b * br) // g
                last = q_start + min(b * br + br - 1, rows - 1) // g
                begin = (max(0, first - window + 1) // split) if window else 0
                items += [0, b, begin, last // split + 1, -1, 0, 0, 0]
        from lockstep_amd.ops import pack_attention_items, pack_combine_items

        items = items * repeat      # the same work many times over (same values to the same places): a full GPU
        seq_row = self.seqs(q_start, t).cpu().numpy()
        n_items = len(items) // 8
        items_t = torch.from_numpy(pack_attention_items(items, seq_row)).to(torch.int32).cuda()
        out = torch.full((t, self.nq * self.d), float("nan"), dtype=self.dtype, device="cuda")
        part_acc = torch.full((max(part_rows, 1), self.d), float("nan"), dtype=torch.float32, device="cuda")
        part_ml = torch.full((max(part_rows, 1), 2), float("nan"), dtype=torch.float32, device="cuda")
        K().attention(qkv, self.nq, self.nkv, self.d, self.k_pages, self.v_pages, self.ps, self.table,
                      self.seqs(q_start, t), items_t, n_items, out, part_acc, part_ml, scale, window,
                      variant, rows, spans=span > 1)
        if combine:
            comb = torch.from_numpy(pack_combine_items(combine, seq_row)).to(torch.int32).cuda()
            K().attention_combine(self.d, self.seqs(q_start, t), comb, len(combine) // 4, self.nq, self.nkv,
                                  part_acc, part_ml, out, max_rows=rows if few_rows else 0)
        return out.view(t, self.nq, self.d)


def rand_qkv(t, nq, nkv, d, dtype, seed, sharp=None):
    g = torch.Generator().manual_seed(seed)
    qkv = torch.randn(t, (nq + 2 * nkv) * d, generator=g)
    if sharp is not None:
        # make one far key stand out for the last query: a fault that drops it shows
        key_pos, = sharp
        q = qkv[:, : nq * d].view(t, nq, d)
        k = qkv[:, nq * d:(nq + nkv) * d].view(t, nkv, d)
        k[key_pos] = q[-1].view(nkv, nq // nkv, d)[:, 0] * 2.0
    return qkv.to(dtype)


def split_qkv(qkv, nq, nkv, d):
    t = qkv.shape[0]
    q = qkv[:, : nq * d].reshape(t, nq, d)
    k = qkv[:, nq * d:(nq + nkv) * d].reshape(t, nkv, d)
    v = qkv[:, (nq + nkv) * d:].reshape(t, nkv, d)
    return q, k, v


ATT_TOL = {torch.float32: 2e-5, torch.bfloat16: 2e-2}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(16, 8, 128, 16), (4, 4, 16, 8), (8, 1, 64, 32), (6, 2, 48, 16),
                                         (32, 4, 80, 64), (2, 2, 256, 128), (64, 8, 128, 16)])
@pytest.mark.parametrize("kv_len", [1, 5, 64, 129, 257, 600])
def test_prefill_attention_matches_naive(dtype, nq, nkv, d, ps, kv_len):
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=kv_len + d)
    case = PagedCase(dtype, nq, nkv, d, ps, kv_len, shuffle_seed=3)
    dev = qkv.cuda()
    case.write(dev, 0)
    out = case.attend(dev, 0, d ** -0.5)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    want = naive_attention(q, k, v, 0, d ** -0.5)
    assert not torch.isnan(out).any()
    assert rel_err(out, want) < ATT_TOL[dtype]
    # the kernel that loads straight from global memory gives the same bits as the LDS-staged one
    assert torch.equal(case.attend(dev, 0, d ** -0.5, variant=1), out)
    if K().wide_supported(d, dtype, ps):
        assert torch.equal(case.attend(dev, 0, d ** -0.5, variant=4), out), "wide kernel"
        assert torch.equal(case.attend(dev, 0, d ** -0.5, variant=5), out), "wide kernel, row blocks of 64"
    if kv_len == 1:
        assert torch.equal(out.cpu().float()[0], v.float()[0].repeat_interleave(nq // nkv, dim=0))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(4, 2, 128, 16), (2, 1, 64, 8), (8, 4, 32, 64)])
def test_attention_over_more_keys_than_one_window_of_page_ids(dtype, nq, nkv, d, ps):
    """A workgroup of the streaming kernels holds the page ids of 32 tiles (4,096 keys) at a time.
    Contexts beyond that: a prompt in one step, late portions and decoded tokens, each walking all
    splits in one workgroup or cut into splits and combined; same bits in every kernel, and the
    32-bit result against the naive formula.  One far key is made to stand out."""
    n = 4096 * 2 + 300
    qkv = rand_qkv(n, nq, nkv, d, dtype, seed=n + d, sharp=(37,))
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=5)
    dev = qkv.cuda()
    case.write(dev, 0)
    full = case.attend(dev, 0, d ** -0.5)                                  # staged or direct kernel, row blocks of 64
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    tail = slice(n - 40, n)
    want = naive_attention(q[tail], k, v, n - 40, d ** -0.5)
    assert rel_err(full[tail], want) < ATT_TOL[dtype]
    if K().wide_supported(d, dtype, ps):
        for variant in (4, 5):
            assert torch.equal(case.attend(dev, 0, d ** -0.5, variant=variant), full), f"wide kernel {variant}"
            late = case.attend(dev[n - 200:], n - 200, d ** -0.5, variant=variant)
            assert torch.equal(late, full[n - 200:]), f"late portion, wide kernel {variant}"
    if K().coop_supported(d, dtype, ps):
        for p in (4095, 4096, 4100, 8191, 8192, n - 1):
            for split in (False, True):
                one = case.attend(dev[p:p + 1], p, d ** -0.5, variant=3, force_split=split)
                assert torch.equal(one, full[p:p + 1]), f"decoded token at {p}, split={split}"
        # with two workgroups a CU the kernel works with one buffer, refilled half by half
        crowd = case.attend(dev[n - 1:], n - 1, d ** -0.5, variant=3, force_split=False, repeat=-(-600 // nkv))
        assert torch.equal(crowd, full[n - 1:]), "decoded token, crowded launch"


@pytest.mark.parametrize("dtype,nq,nkv,d,ps", [(torch.bfloat16, 4, 2, 256, 16), (torch.bfloat16, 4, 2, 128, 8),
                                               (torch.float32, 4, 2, 128, 8), (torch.float32, 2, 1, 80, 16)])
def test_wide_attention_at_the_edges_of_its_row_blocks_and_page_windows(dtype, nq, nkv, d, ps):
    """Portions whose rows end beside a wave's, a workgroup's and a large block's edge, over contexts that end beside a
    tile's edge and beside a window of page ids': the bits of the kernel that loads straight from global memory."""
    starts, lengths = (0, 127, 4000), (31, 32, 33, 63, 64, 65, 95, 96, 97, 130)
    n = max(starts) + max(lengths)
    qkv = rand_qkv(n, nq, nkv, d, dtype, seed=d + ps)
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=7)
    dev = qkv.cuda()
    case.write(dev, 0)
    assert K().wide_supported(d, dtype, ps)
    for start in starts:
        for length in lengths:
            rows = dev[start:start + length]
            want = case.attend(rows, start, d ** -0.5, variant=1, force_split=False)
            for variant in (4, 5):
                got = case.attend(rows, start, d ** -0.5, variant=variant, force_split=False)
                assert torch.equal(got, want), (start, length, variant)


@pytest.mark.parametrize("dtype,nq,nkv,d,ps", [(torch.bfloat16, 4, 2, 112, 16), (torch.bfloat16, 3, 1, 144, 8), (torch.float32, 4, 2, 144, 16),
                                               (torch.float32, 3, 1, 112, 128), (torch.bfloat16, 4, 2, 160, 64), (torch.bfloat16, 2, 2, 192, 8)])
@pytest.mark.parametrize("window", [0, 150])
def test_wide_attention_where_a_load_spans_several_pages(dtype, nq, nkv, d, ps, window):
    """Head sizes whose rows do not divide a wave's load: every lane looks its piece's page up, among the sixteen of a tile, and
    the last round of loads is only some waves'.  The bits of the kernel that loads straight from global memory."""
    n = 4000 + 130
    qkv = rand_qkv(n, nq, nkv, d, dtype, seed=d + ps)
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=9)
    dev = qkv.cuda()
    case.write(dev, 0)
    assert K().wide_supported(d, dtype, ps)
    for start, length in ((0, 97), (127, 65), (4000, 130), (3967, 33)):
        rows = dev[start:start + length]
        want = case.attend(rows, start, d ** -0.5, window=window, variant=1, force_split=False)
        for variant in (4, 5):
            got = case.attend(rows, start, d ** -0.5, window=window, variant=variant, force_split=False)
            assert torch.equal(got, want), (start, length, variant)


@pytest.mark.parametrize("dtype,largest_shared", [(torch.bfloat16, 144), (torch.float32, 64)])
def test_wide_attention_has_eight_waves_where_a_workgroup_has_the_cu(dtype, largest_shared):
    """Two workgroups' tiles and page ids fit a CU's 160 KB up to these head sizes."""
    for d in (16, 32, 48, 64, 80, 112, 128, 144, 160, 192, 256):
        if K().wide_supported(d, dtype, 16):
            assert K().wide_eight_waves(d, dtype) == (d > largest_shared), d


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(16, 8, 128, 16), (6, 3, 32, 8), (8, 1, 64, 16)])
def test_attention_row_is_the_same_alone_in_a_portion_and_in_the_whole_prompt(dtype, nq, nkv, d, ps):
    """A query row alone (decode, split mode), in a portion, and in a whole prefill: same bits;
    also under a shuffled block table."""
    kv_len = 700
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=11, sharp=(3,)).cuda()
    whole = PagedCase(dtype, nq, nkv, d, ps, kv_len)
    whole.write(qkv, 0)
    full = whole.attend(qkv, 0, d ** -0.5)
    shuffled = PagedCase(dtype, nq, nkv, d, ps, kv_len, shuffle_seed=99)
    shuffled.write(qkv, 0)
    assert torch.equal(shuffled.attend(qkv, 0, d ** -0.5), full)
    for p in (0, 1, 15, 16, 17, 127, 128, 255, 256, 257, 511, 512, 699):
        alone = whole.attend(qkv[p:p + 1], p, d ** -0.5)
        assert torch.equal(alone[0], full[p]), f"row {p} alone"
        alone = whole.attend(qkv[p:p + 1], p, d ** -0.5, variant=1)
        assert torch.equal(alone[0], full[p]), f"row {p} alone, loaded directly"
        if K().coop_supported(d, dtype, ps):
            for split in (True, False):
                alone = whole.attend(qkv[p:p + 1], p, d ** -0.5, variant=3, force_split=split)
                assert torch.equal(alone[0], full[p]), f"row {p} alone, cooperative kernel, split={split}"
        both = whole.attend(qkv[p:p + 1], p, d ** -0.5, force_split=False)
        assert torch.equal(both[0], full[p]), f"row {p} alone, direct"
    for lo, hi in ((250, 262), (0, 3), (500, 700), (255, 257), (690, 700)):
        part = whole.attend(qkv[lo:hi], lo, d ** -0.5)
        assert torch.equal(part, full[lo:hi]), f"portion {lo}:{hi}"
        part = whole.attend(qkv[lo:hi], lo, d ** -0.5, force_split=True)
        assert torch.equal(part, full[lo:hi]), f"portion {lo}:{hi} split"
        if K().wide_supported(d, dtype, ps):
            for variant in (4, 5):
                for split in (False, True):
                    part = whole.attend(qkv[lo:hi], lo, d ** -0.5, variant=variant, force_split=split)
                    assert torch.equal(part, full[lo:hi]), f"portion {lo}:{hi}, wide kernel {variant}, split={split}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps,t", [(4, 1, 128, 16, 300), (4, 2, 64, 8, 517), (6, 3, 128, 64, 260), (8, 4, 128, 32, 530),
                                           (16, 8, 64, 16, 129), (16, 16, 128, 128, 140), (24, 24, 16, 16, 90)])
def test_row_blocks_of_every_number_of_kv_heads_with_scales_of_either_sign_and_windows(dtype, nq, nkv, d, ps, t):
    """How the work of a portion is numbered depends on the kv heads and on the row blocks (here odd and even
    counts): the wide kernels against the direct one, to the bit, and against the formula.  A negative scale
    turns the order of the scores, a zero one makes them equal; a window releases the pages behind it."""
    n = 700
    qkv = rand_qkv(n, nq, nkv, d, dtype, seed=nq + d)
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=7)
    dev = qkv.cuda()
    case.write(dev, 0)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    lo = n - t
    for scale, window in ((d ** -0.5, 0), (-0.7 * d ** -0.5, 0), (0.0, 0), (d ** -0.5, 131)):
        saved = case.table.clone()
        if window:
            case.table[1, :max(0, lo - window + 1) // ps] = -1
        got = case.attend(dev[lo:], lo, scale, window=window, variant=1, force_split=False)
        want = naive_attention(q[lo:], k, v, lo, scale, window=window or None)
        assert rel_err(got, want) < ATT_TOL[dtype], (scale, window)
        if K().wide_supported(d, dtype, ps):
            for variant in (4, 5):
                for split in (False, True):
                    wide = case.attend(dev[lo:], lo, scale, window=window, variant=variant, force_split=split)
                    assert torch.equal(wide, got), (scale, window, variant, split)
        case.table.copy_(saved)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 7, 128, 300])
def test_attention_window(dtype, window):
    nq, nkv, d, ps, kv_len = 4, 2, 32, 16, 520
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=window, sharp=(kv_len - window,))
    case = PagedCase(dtype, nq, nkv, d, ps, kv_len)
    dev = qkv.cuda()
    case.write(dev, 0)
    out = case.attend(dev, 0, d ** -0.5, window=window)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    want = naive_attention(q, k, v, 0, d ** -0.5, window=window)
    assert rel_err(out, want) < ATT_TOL[dtype]
    assert torch.equal(case.attend(dev, 0, d ** -0.5, window=window, variant=1), out)
    assert torch.equal(case.attend(dev, 0, d ** -0.5, window=window, variant=4), out)
    assert torch.equal(case.attend(dev, 0, d ** -0.5, window=window, variant=5), out)
    # pages behind the window may be gone: mark them released and decode the last rows
    for p in (kv_len - 1, 300, 130):
        first_needed = max(0, p - window + 1) // ps
        saved = case.table.clone()
        case.table[1, :first_needed] = -1
        alone = case.attend(dev[p:p + 1], p, d ** -0.5, window=window)
        coop = case.attend(dev[p:p + 1], p, d ** -0.5, window=window, variant=3)
        case.table.copy_(saved)
        lo = max(0, p - 70)                     # a portion: what its first row needs must be held
        case.table[1, :max(0, lo - window + 1) // ps] = -1
        wide = case.attend(dev[lo:p + 1], lo, d ** -0.5, window=window, variant=4)
        case.table.copy_(saved)
        assert torch.equal(alone[0], out[p]), f"row {p}"
        assert torch.equal(coop[0], out[p]), f"row {p}, cooperative kernel"
        assert torch.equal(wide, out[lo:p + 1]), f"rows {lo}..{p}, wide kernel"


def test_more_row_blocks_than_a_grid_numbers_in_its_second_dimension():
    """The same three row blocks 22,000 times over (65,535 a launch): all are worked on, the last launch's too."""
    n, nq, nkv, d = 70, 4, 2, 16
    qkv = rand_qkv(n, nq, nkv, d, torch.bfloat16, seed=1)
    case = PagedCase(torch.bfloat16, nq, nkv, d, 16, n, shuffle_seed=7)
    case.write(qkv.cuda(), 0)
    want = case.attend(qkv.cuda(), 0, 0.25, variant=1, force_split=False)
    assert torch.equal(case.attend(qkv.cuda(), 0, 0.25, variant=5, force_split=False, repeat=22000), want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(4, 2, 64, 16), (16, 8, 128, 16), (6, 2, 48, 8)])
@pytest.mark.parametrize("scale", [0.13, -0.13])
def test_scores_of_great_size_leave_finite_results(dtype, nq, nkv, d, ps, scale):
    """Queries and keys of +-2^20 and scores up to 10^13: the largest probability of a row is exp(0) whatever its score, so
    nothing overflows.  Products and sums are whole multiples of 2^40 below 2^47 and exact in every order, so equal scores tie
    exactly, and a step between two scores (2^41 times the scale) leaves the lower one nothing."""
    n = 700
    g = torch.Generator().manual_seed(d)
    qkv = torch.randn(n, (nq + 2 * nkv) * d, generator=g)
    signs = torch.randint(0, 2, (n, (nq + nkv) * d), generator=g).float() * 2 - 1
    qkv[:, : (nq + nkv) * d] = signs * 2.0 ** 20
    qkv = qkv.to(dtype)
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=2)
    dev = qkv.cuda()
    case.write(dev, 0)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    want = naive_attention(q, k, v, 0, scale)
    for variant in (0, 1) + ((4, 5) if K().wide_supported(d, dtype, ps) else ()):
        got = case.attend(dev, 0, scale, variant=variant, force_split=False)
        assert torch.isfinite(got).all(), variant
        assert rel_err(got, want) < ATT_TOL[dtype], variant
    for p in (5, 127, 128, n - 1):
        for split in (False, True):
            one = case.attend(dev[p:p + 1], p, scale, variant=3, force_split=split)
            assert torch.isfinite(one).all() and rel_err(one, want[p:p + 1]) < ATT_TOL[dtype], (p, split)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(4, 2, 64, 16), (16, 8, 128, 16), (6, 2, 48, 8)])
@pytest.mark.parametrize("largest", [0.95 * 2.0 ** 128, -0.95e30])
def test_scores_at_the_ends_of_their_range(dtype, nq, nkv, d, ps, largest):
    """Scores close to the largest float32, and scores close above the -1e30 that running maxima start at: they are finite as
    they are, so they are not to be multiplied by a constant beyond 1 before the row's largest is taken off.  Queries are 2^60 in
    every element and keys +-2^60, so every partial sum is a whole multiple of 2^120 that float32 holds exactly in any order."""
    n = 300
    g = torch.Generator().manual_seed(d)
    qkv = torch.randn(n, (nq + 2 * nkv) * d, generator=g)
    keys = torch.full((n, nkv, d), 2.0 ** 60)
    for i in range(n):
        for h in range(nkv):         # (up to an eighth of the elements turned: scores from 3/4 of the largest size on)
            turned = int(torch.randint(0, d // 8 + 1, (1,), generator=g))
            keys[i, h, torch.randperm(d, generator=g)[:turned]] *= -1.0
    qkv[:, : nq * d] = 2.0 ** 60
    qkv[:, nq * d:(nq + nkv) * d] = keys.flatten(1)
    qkv = qkv.to(dtype)
    scale = largest / (d * 2.0 ** 120)
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=2)
    dev = qkv.cuda()
    case.write(dev, 0)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    want = naive_attention(q, k, v, 0, scale)
    for variant in (0, 1) + ((4, 5) if K().wide_supported(d, dtype, ps) else ()):
        got = case.attend(dev, 0, scale, variant=variant, force_split=False)
        assert torch.isfinite(got).all() and rel_err(got, want) < ATT_TOL[dtype], variant
    for p in (0, 5, 127, 128, n - 1):
        for split in (False, True):
            one = case.attend(dev[p:p + 1], p, scale, variant=3, force_split=split)
            assert torch.isfinite(one).all() and rel_err(one, want[p:p + 1]) < ATT_TOL[dtype], (p, split)


@pytest.mark.parametrize("nq,nkv,d,ps", [(4, 2, 64, 16), (16, 8, 128, 16), (6, 2, 48, 8), (2, 1, 256, 32)])
def test_rows_of_great_scores_beside_others(nq, nkv, d, ps):
    """Rows whose largest scores lie from 300 to 3,000, side by side: every kernel gives a row the same bits, alone or among the
    others, walked or folded from splits, and they are right."""
    n, dtype, scale = 300, torch.bfloat16, d ** -0.5
    g = torch.Generator().manual_seed(d + nq)
    along = torch.nn.functional.normalize(torch.randn(d, generator=g), dim=0)
    qkv = torch.randn(n, (nq + 2 * nkv) * d, generator=g)
    tops = 300.0 * 10.0 ** torch.rand(n, nq, 1, generator=g)
    q, k = qkv[:, : nq * d].view(n, nq, d), qkv[:, nq * d:(nq + nkv) * d].view(n, nkv, d)
    q += along * tops / (32.0 * scale)
    k *= 0.1
    k += along * 32.0
    qkv = qkv.to(dtype)
    case = PagedCase(dtype, nq, nkv, d, ps, n, shuffle_seed=4)
    dev = qkv.cuda()
    case.write(dev, 0)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    want = naive_attention(q, k, v, 0, scale)
    out = case.attend(dev, 0, scale, variant=1, force_split=False)
    assert rel_err(out, want) < ATT_TOL[dtype]
    for variant in (0,) + ((4, 5) if K().wide_supported(d, dtype, ps) else ()):
        assert torch.equal(case.attend(dev, 0, scale, variant=variant, force_split=False), out), variant
    for p in (0, 127, 128, 200, n - 1):
        for split in (False, True):
            assert torch.equal(case.attend(dev[p:p + 1], p, scale, variant=3, force_split=split), out[p:p + 1]), (p, split)


@pytest.mark.parametrize("dtype", DTYPES)
def test_norm_rotation_and_cache_write(dtype):
    nq, nkv, d, ps, t, start = 6, 3, 32, 8, 21, 5
    rot = 32
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(t, (nq + 2 * nkv) * d, generator=g).to(dtype)
    qw = 1 + 0.2 * torch.randn(d, generator=g)
    kw = 1 + 0.2 * torch.randn(d, generator=g)
    eps, theta = 1e-5, 1e4
    pos = torch.arange(64, dtype=torch.float64)
    inv = 1.0 / (theta ** (torch.arange(0, rot // 2, dtype=torch.float64) * 2 / rot))
    ang = pos[:, None] * inv[None, :]
    cos, sin = ang.cos().float(), ang.sin().float()
    case = PagedCase(dtype, nq, nkv, d, ps, start + t, shuffle_seed=1)
    dev = qkv.clone().cuda()
    case.write(dev, start, qw.cuda(), kw.cuda(), eps, cos.cuda(), sin.cuda(), rot)

    q, k, v = split_qkv(qkv.double(), nq, nkv, d)

    def norm_rope(x, w):
        x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()
        c = cos[start:start + t].double()[:, None, :]
        s = sin[start:start + t].double()[:, None, :]
        lo, hi = x[..., : rot // 2], x[..., rot // 2:rot]
        return torch.cat([lo * c - hi * s, hi * c + lo * s, x[..., rot:]], dim=-1)

    tol = 1e-6 if dtype is torch.float32 else 8e-3
    got_q = dev[:, : nq * d].view(t, nq, d)
    assert rel_err(got_q, norm_rope(q, qw)) < tol
    table = case.table[1].cpu()
    want_k = norm_rope(k, kw)
    for i in range(t):
        p = start + i
        page, slot = int(table[p // ps]), p % ps
        assert rel_err(case.k_pages[page, :, slot, :], want_k[i]) < tol
        assert torch.equal(case.v_pages[page, :, :, slot].cpu().double(), v[i])
    # position 0 leaves a head untouched by the rotation (cos 1, sin 0)
    case0 = PagedCase(dtype, nq, nkv, d, ps, 1)
    one = qkv[:1].clone().cuda()
    case0.write(one, 0, None, None, eps, cos.cuda(), sin.cuda(), rot)
    assert torch.equal(one.cpu(), qkv[:1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(16, 8, 128, 16), (4, 4, 16, 8), (8, 1, 64, 32), (6, 2, 48, 16),
                                         (32, 2, 80, 64), (2, 2, 256, 128), (3, 3, 32, 8), (64, 8, 128, 16)])
def test_decode_attention_is_the_same_in_every_kernel(dtype, nq, nkv, d, ps):
    """The last one or two tokens of a sequence through the staged, the direct
    and the cooperative kernel, split or not: same bits, and right."""
    kv_len = 700
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=d + nq, sharp=(5,))
    case = PagedCase(dtype, nq, nkv, d, ps, kv_len, shuffle_seed=7)
    dev = qkv.cuda()
    case.write(dev, 0)
    q, k, v = split_qkv(qkv.double(), nq, nkv, d)
    want = naive_attention(q, k, v, 0, d ** -0.5)
    g = nq // nkv
    for start, n in ((699, 1), (698, 2), (255, 1), (256, 1), (0, 1), (127, 2)):
        if n * g > 16:
            n = 1
        ref = case.attend(dev[start:start + n], start, d ** -0.5, variant=1, force_split=False)
        assert rel_err(ref, want[start:start + n]) < ATT_TOL[dtype], (start, n)
        variants = [(0, True), (0, False), (1, True)]
        if K().coop_supported(d, dtype, ps):
            variants += [(3, True), (3, False)]
        if K().wide_supported(d, dtype, ps):
            variants += [(4, True), (4, False)]
        for variant, split in variants:
            got = case.attend(dev[start:start + n], start, d ** -0.5, variant=variant, force_split=split)
            assert torch.equal(got, ref), f"start={start} n={n} variant={variant} split={split}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(16, 8, 128, 16), (4, 4, 16, 8), (6, 2, 48, 16), (3, 3, 32, 8),
                                         (64, 8, 128, 16)])
def test_cooperative_items_of_several_splits_leave_the_same_partial_results(dtype, nq, nkv, d, ps):
    """A long request cut into work items of one, two, three or four splits each (a partial result a
    split, folded by the combine kernel), laid out for more splits than it has, with and without
    a window: the bits of one workgroup walking the whole request."""
    if not K().coop_supported(d, dtype, ps):
        pytest.skip("the cooperative kernel's tiles do not fit")
    kv_len = 1400                                     # six splits, the last one partly filled
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=3 * d + nq, sharp=(9,))
    case = PagedCase(dtype, nq, nkv, d, ps, kv_len, shuffle_seed=5)
    dev = qkv.cuda()
    case.write(dev, 0)
    for window in (0, 700):
        for start in (1399, 1279, 1024, 511):
            ref = case.attend(dev[start:start + 1], start, d ** -0.5, window=window, variant=3, force_split=False)
            for span, pad in ((1, 0), (2, 0), (3, 1), (4, 0), (4, 3), (8, 0)):
                for few in (False, True):
                    got = case.attend(dev[start:start + 1], start, d ** -0.5, window=window, variant=3,
                                      force_split=True, span=span, pad_splits=pad, few_rows=few)
                    assert torch.equal(got, ref), f"start={start} window={window} span={span} pad={pad} few={few}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps", [(16, 8, 128, 16), (4, 4, 16, 8), (6, 2, 48, 16), (2, 1, 256, 16),
                                         (64, 8, 128, 16)])
def test_the_fold_for_few_rows_has_the_bits_of_the_general_fold_over_many_splits(dtype, nq, nkv, d, ps):
    """Forty-one splits (more than two of the fold's rounds of sixteen), one and three tokens."""
    if not K().coop_supported(d, dtype, ps):
        pytest.skip("the cooperative kernel's tiles do not fit")
    kv_len = 256 * 40 + 77
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=5 * d + nq, sharp=(300,))
    case = PagedCase(dtype, nq, nkv, d, ps, kv_len, shuffle_seed=6)
    dev = qkv.cuda()
    case.write(dev, 0)
    for tokens in (1, 3):
        if tokens * (nq // nkv) > 16:
            continue
        start = kv_len - tokens
        ref = case.attend(dev[start:], start, d ** -0.5, variant=3, force_split=False)
        for span in (1, 5):
            general = case.attend(dev[start:], start, d ** -0.5, variant=3, force_split=True, span=span)
            few = case.attend(dev[start:], start, d ** -0.5, variant=3, force_split=True, span=span, few_rows=True)
            assert torch.equal(general, ref) and torch.equal(few, ref), f"tokens={tokens} span={span}"


@pytest.mark.parametrize("dtype", DTYPES)
def test_the_fold_for_few_rows_is_right_when_it_is_handed_more_rows_than_it_was_promised(dtype):
    """The caller says "at most 16 rows" and a request brings 24 and 40: the fold notices and takes the
    general way (it used to leave the rows beyond the sixteenth unwritten)."""
    nq, nkv, d, ps = 8, 1, 64, 16
    kv_len = 900
    qkv = rand_qkv(kv_len, nq, nkv, d, dtype, seed=77, sharp=(40,))
    case = PagedCase(dtype, nq, nkv, d, ps, kv_len, shuffle_seed=2)
    dev = qkv.cuda()
    case.write(dev, 0)
    for tokens in (3, 5):
        start = kv_len - tokens
        ref = case.attend(dev[start:], start, d ** -0.5, variant=0, force_split=False)
        lied = case.attend(dev[start:], start, d ** -0.5, variant=0, force_split=True, few_rows=True)
        assert not torch.isnan(lied).any() and torch.equal(lied, ref), tokens


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps,rot,normed,window", [
    (16, 8, 128, 16, 128, True, 0), (64, 8, 128, 16, 128, True, 0), (8, 1, 64, 32, 64, True, 0), (4, 4, 16, 8, 16, True, 0),
    # sixteen query heads a kv head: with the new key and value more heads than a workgroup has groups of sixteen lanes
    (16, 1, 64, 16, 64, True, 0), (30, 2, 32, 8, 16, True, 0),
    (6, 2, 48, 16, 32, False, 0), (4, 2, 32, 8, 0, True, 0), (4, 2, 64, 16, 64, True, 200)])
def test_fused_decode_attention_equals_the_separate_kernels(dtype, nq, nkv, d, ps, rot, normed, window):
    """A decoded token through qk_rope_kv + cooperative attention, and through the one fused launch:
    the same output bits and the same cache contents, at the edges of pages, tiles and splits."""
    if not K().decode_fused_supported(d, dtype, ps):
        pytest.skip("the fused decode kernel does not fit into LDS for this head size")
    from lockstep_amd.ops import kernels

    g = torch.Generator().manual_seed(d + nq)
    total = 530
    qkv = (torch.randn(total, (nq + 2 * nkv) * d, generator=g) * 2).to(dtype).cuda()
    qw = (1 + 0.3 * torch.randn(d, generator=g)).cuda() if normed else None
    kw = (1 + 0.3 * torch.randn(d, generator=g)).cuda() if normed else None
    cos = sin = None
    if rot:
        inv = 1.0 / (1e4 ** (torch.arange(0, rot // 2, dtype=torch.float64) * 2 / rot))
        ang = torch.arange(total, dtype=torch.float64)[:, None] * inv[None, :]
        cos, sin = ang.cos().float().cuda(), ang.sin().float().cuda()
    eps = 1e-5
    tile, split = kernels().attention_geometry(d)
    for p in (0, 1, ps - 1, ps, 127, 128, 255, 256, 257, 300, 511, 512, 529):
        base = PagedCase(dtype, nq, nkv, d, ps, p + 1, shuffle_seed=p)
        if p:
            ctx_rows = qkv[:p].clone()
            base.write(ctx_rows, 0, qw, kw, eps, cos, sin, rot)
        first_needed = max(0, p - window + 1) // ps if window else 0
        base.table[1, :first_needed] = -1
        k0, v0 = base.k_pages.clone(), base.v_pages.clone()
        # separate kernels
        row = qkv[p:p + 1].clone()
        base.write(row, p, qw, kw, eps, cos, sin, rot)
        want = base.attend(row, p, d ** -0.5, window=window, variant=3)
        k_want, v_want = base.k_pages.clone(), base.v_pages.clone()
        for use_split in (True, False):
            base.k_pages.copy_(k0); base.v_pages.copy_(v0)
            lo = max(0, p - window + 1) if window else 0
            split_lo = lo // split
            n_splits = p // split + 1 - split_lo
            if use_split:
                items = [v for s_ in range(split_lo, split_lo + n_splits) for v in (0, 0, s_, s_ + 1, 0, n_splits, split_lo, 0)]
                combine = [0, 0, 0, n_splits]
            else:
                items, combine = [0, 0, split_lo, p // split + 1, -1, 0, 0, 0], []
            part_rows = max(nkv * (nq // nkv) * n_splits, 1)
            part_acc = torch.full((part_rows, d), float("nan"), dtype=torch.float32, device="cuda")
            part_ml = torch.full((part_rows, 2), float("nan"), dtype=torch.float32, device="cuda")
            out = torch.full((1, nq * d), float("nan"), dtype=dtype, device="cuda")
            from lockstep_amd.ops import pack_attention_items, pack_combine_items

            seq_row = base.seqs(p, 1).cpu().numpy()
            # the items of one tile once as they are and once with the tile's page ids inside them
            one_tile = split == tile and all(items[i + 3] - items[i + 2] == 1 for i in range(0, len(items), 8))
            for with_pages in (False, True) if one_tile and tile // ps <= 16 else (False,):
                base.k_pages.copy_(k0); base.v_pages.copy_(v0)
                part_acc.fill_(float("nan")); part_ml.fill_(float("nan")); out.fill_(float("nan"))
                ids = None
                if with_pages:
                    row_of_table = base.table[int(seq_row.reshape(-1, 8)[0, 4])].cpu().numpy()
                    ids = np.full((len(items) // 8, 16), -1, dtype=np.int64)
                    for i in range(len(items) // 8):
                        held = row_of_table[items[8 * i + 2] * (tile // ps):][: tile // ps]
                        ids[i, : len(held)] = held
                items_t = torch.from_numpy(pack_attention_items(items, seq_row, ids)).to(torch.int32).cuda()
                raw = qkv[p:p + 1].clone()
                K().attention_decode(raw, nq, nkv, d, base.k_pages, base.v_pages, ps, base.table, base.seqs(p, 1),
                                     items_t, len(items) // 8, out, part_acc, part_ml, d ** -0.5, window, qw, kw, eps,
                                     cos, sin, rot, p, True, single_tile=one_tile)
                if combine:
                    comb = torch.from_numpy(pack_combine_items(combine, seq_row)).to(torch.int32).cuda()
                    K().attention_combine(d, base.seqs(p, 1), comb, 1, nq, nkv, part_acc, part_ml, out)
                what = f"position {p}, split={use_split}, page ids in the items: {with_pages}"
                assert torch.equal(out.view(1, nq, d), want), what
                same_k = (base.k_pages == k_want) | ((base.k_pages != base.k_pages) & (k_want != k_want))
                same_v = (base.v_pages == v_want) | ((base.v_pages != base.v_pages) & (v_want != v_want))
                assert bool(same_k.all()) and bool(same_v.all()), f"cache after {what}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m", [1, 9, 16, 40, 200])
@pytest.mark.parametrize("inter,k", [(136, 96), (3072, 1024), (48, 260)])
def test_gemm_with_swiglu_epilogue(dtype, m, inter, k):
    """Gate and up interleaved in tiles of 16 rows, activation in the epilogue:
    equals silu(x Wg^T) * (x Wu^T); a row has the same bits at any batch size."""
    from lockstep_amd.ops import SWIGLU, interleave_gate_up

    g = torch.Generator().manual_seed(inter + k)
    x = torch.randn(m, k, generator=g).to(dtype)
    gate = (torch.randn(inter, k, generator=g) * 0.2).to(dtype)
    up = (torch.randn(inter, k, generator=g) * 0.2).to(dtype)
    w = interleave_gate_up(gate, up).cuda()
    assert w.shape[0] % 32 == 0 and torch.equal(w[16:32, :].cpu(), up[:16])
    out = torch.empty(m, inter, dtype=dtype, device="cuda")
    K().gemm(x.cuda(), w, out, SWIGLU)
    want = torch.nn.functional.silu(x.double() @ gate.double().T) * (x.double() @ up.double().T)
    assert rel_err(out, want) < TOL[dtype]
    one = torch.empty(1, inter, dtype=dtype, device="cuda")
    K().gemm(x[m - 1:].cuda(), w, one, SWIGLU)
    assert torch.equal(one[0], out[m - 1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(1, 64, 1024), (8, 272, 96), (16, 100, 3072), (5, 48, 200)])
def test_gemm_with_fused_norm_equals_norm_then_gemm(dtype, m, n, k):
    """The RMSNorm prologue of the skinny kernel gives the bits of the
    stand-alone norm kernel followed by the plain product, also with the
    SwiGLU epilogue."""
    from lockstep_amd.ops import STORE, SWIGLU, interleave_gate_up

    g = torch.Generator().manual_seed(m + n + k)
    h = (torch.randn(m, k, generator=g) * 3).cuda()
    nw = (1 + 0.2 * torch.randn(k, generator=g)).cuda()
    w = (torch.randn(n, k, generator=g) * 0.1).to(dtype).cuda()
    eps = 1e-5
    normed = torch.empty(m, k, dtype=dtype, device="cuda")
    K().rmsnorm(h, nw, normed, eps)
    want = torch.empty(m, n, dtype=dtype, device="cuda")
    K().gemm(normed, w, want, STORE)
    got = torch.empty(m, n, dtype=dtype, device="cuda")
    K().gemm(h, w, got, STORE, norm_weight=nw, eps=eps)
    assert torch.equal(got, want)
    inter = n // 2
    wi = interleave_gate_up(w[:inter].cpu(), w[inter:2 * inter].cpu()).cuda()
    want2 = torch.empty(m, inter, dtype=dtype, device="cuda")
    K().gemm(normed, wi, want2, SWIGLU)
    got2 = torch.empty(m, inter, dtype=dtype, device="cuda")
    K().gemm(h, wi, got2, SWIGLU, norm_weight=nw, eps=eps)
    assert torch.equal(got2, want2)
    from lockstep_amd.ops import KernelError
    with pytest.raises(KernelError):
        K().gemm(torch.zeros(17, k, device="cuda"), w, torch.empty(17, n, dtype=dtype, device="cuda"), STORE,
                 norm_weight=nw, eps=eps)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m", [1, 8, 16, 17, 40, 64, 65, 100, 200, 256])
@pytest.mark.parametrize("n,k", [(1024, 3072), (96, 520), (1024, 2048), (40, 64), (4096, 1024), (5120, 96),
                                 (1028, 4096), (16384, 64), (16388, 64),
                                 # enough column blocks and slices that workgroups walk several blocks
                                 (4104, 4096), (4104, 12288), (4200, 8192), (8200, 2048),
                                 # K of 25,600: fifteen slices of 1,792 (the last one shorter)
                                 (5120, 25600), (1032, 25600)])
def test_slice_sums_and_fused_add_norm_equal_the_separate_kernels(dtype, m, n, k):
    """gemm_slices + add_rmsnorm give the bits of gemm(ADD_F32) + rmsnorm: the residual row and the
    normalised row; also for a list of rows and for the plain addition.  More than 64 rows (several
    groups of rows walking the same weights) where the slice length has such a kernel; elsewhere the
    product says so."""
    from lockstep_amd.ops import ADD_F32

    most = K().gemm_slices_max_rows(k, dtype)
    assert most in (64, 256) and (most == 256) == (k <= (8192 if dtype is torch.bfloat16 else 4096))
    if m > most:
        with pytest.raises(RuntimeError, match="gemm_slices"):
            K().gemm_slices(torch.zeros(m, k, dtype=dtype, device="cuda"), torch.zeros(n, k, dtype=dtype, device="cuda"),
                            torch.zeros(K().gemm_slices_count(k), m, n, device="cuda"))
        return
    g = torch.Generator().manual_seed(n + k + m)
    x = torch.randn(m, k, generator=g).to(dtype).cuda()
    w = (torch.randn(n, k, generator=g) * 0.1).to(dtype).cuda()
    h0 = torch.randn(m, n, generator=g).cuda()
    weight = (1 + 0.1 * torch.randn(n, generator=g)).cuda()
    eps = 1e-5
    h_ref = h0.clone()
    K().gemm(x, w, h_ref, ADD_F32)
    y_ref = torch.empty(m, n, dtype=dtype, device="cuda")
    K().rmsnorm(h_ref, weight, y_ref, eps)
    slices = K().gemm_slices_count(k)
    partials = torch.full((slices, m, n), float("nan"), device="cuda")
    K().gemm_slices(x, w, partials)
    assert not torch.isnan(partials).any()
    h = h0.clone()
    y = torch.empty(m, n, dtype=dtype, device="cuda")
    K().add_rmsnorm(h, partials, weight, y, eps)
    assert torch.equal(h, h_ref) and torch.equal(y, y_ref)
    want = (h0.double() + x.double() @ w.double().T)
    assert rel_err(h, want) < (1e-5 if dtype is torch.float32 else 2e-2)
    h = h0.clone()
    K().add_rmsnorm(h, partials, None, None)
    assert torch.equal(h, h_ref)
    rows = torch.tensor([m - 1, 0][: min(2, m)], dtype=torch.int32).cuda()
    h = h0.clone()
    y = torch.empty(rows.shape[0], n, dtype=dtype, device="cuda")
    K().add_rmsnorm(h, partials, weight, y, eps, rows)
    assert torch.equal(y, y_ref[rows.long()])
    assert torch.equal(h[rows.long()], h_ref[rows.long()])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,nq,nkv,d,n,splits", [(1, 16, 8, 128, 1024, 3), (8, 16, 8, 128, 1024, 4), (16, 4, 2, 64, 520, 2),
                                                 (5, 32, 8, 128, 4096, 8), (3, 6, 3, 32, 96, 5), (2, 64, 8, 128, 5120, 2),
                                                 (7, 2, 1, 256, 300, 3)])
def test_the_product_that_folds_the_splits_itself_equals_fold_then_product(dtype, m, nq, nkv, d, n, splits):
    """The per-split sums of m decoded tokens (some splits empty, with NaN where nothing may be read; one
    token with nothing but empty splits) through the combine launch and ``gemm_slices``, and through
    ``gemm_slices_folded`` alone: the same slice sums, bit for bit."""
    from lockstep_amd.ops import pack_combine_items

    k = nq * d
    if not K().gemm_slices_folded_ok(dtype, m, n, k, d, splits):
        assert dtype is torch.float32 or n * k * 2 >= 64 << 20, "refused although the plain slice kernel would run"
        pytest.skip("the folded product does not take these sizes")
    g = torch.Generator().manual_seed(m * 100 + nq + d + splits)
    rows = m * nq * splits
    acc = torch.randn(rows, d, generator=g) * 3
    ml = torch.stack([torch.randn(rows, generator=g) * 4, torch.rand(rows, generator=g) * 50 + 0.01], dim=1)
    empty = torch.rand(rows, generator=g) < 0.25
    empty.view(m, nq, splits)[m - 1] = True                     # the last token saw no key at all
    ml[empty, 0], ml[empty, 1] = -1e30, 0.0
    acc[empty] = float("nan")
    acc, ml = acc.cuda(), ml.cuda()
    w = (torch.randn(n, k, generator=g) * 0.1).to(dtype).cuda()
    seqs = torch.tensor([[i, 1, 700 + i, 701 + i, i, 0, 0, 0] for i in range(m)], dtype=torch.int32)
    items = torch.from_numpy(pack_combine_items([(i, 0, i * nq * splits, splits) for i in range(m)], seqs.numpy())).to(torch.int32)
    attn = torch.full((m, k), float("nan"), dtype=dtype, device="cuda")
    K().attention_combine(d, seqs.cuda(), items.cuda(), m, nq, nkv, acc, ml, attn, max_rows=nq // nkv)
    assert not torch.isnan(attn).any() and (attn[m - 1] == 0).all()
    slices = K().gemm_slices_count(k)
    want = torch.full((slices, m, n), float("nan"), device="cuda")
    K().gemm_slices(attn, w, want)
    got = torch.full((slices, m, n), float("nan"), device="cuda")
    K().gemm_slices_folded(acc, ml, splits, d, w, got)
    assert not torch.isnan(got).any()
    assert torch.equal(got, want)
    # and right: against the fold in float64
    a, b = acc.cpu().double().view(m, nq, splits, d), ml.cpu().double().view(m, nq, splits, 2)
    a[b[..., 1] <= 0] = 0
    top = b[..., 0].max(dim=2, keepdim=True).values
    scale = torch.where(b[..., 1] > 0, (b[..., 0] - top).exp(), torch.zeros_like(top))
    total = (b[..., 1] * scale).sum(2)
    x = (a * scale[..., None]).sum(2) / total.clamp_min(1e-300)[..., None]
    x[total <= 0] = 0
    product = x.reshape(m, k) @ w.cpu().double().T
    assert rel_err(got.sum(0), product) < (1e-4 if dtype is torch.float32 else 2e-2)
