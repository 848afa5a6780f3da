"""The tile kernels on 16-bit and packed 4-bit weights: every tile height at the edges of its row fragments (which are skipped past an
expert's rows) and of the tile, against a float32 product of the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 0, 95, 96, 97, 33, 127, 128, 129, 191, 192, 193, 400]


@pytest.mark.parametrize("variant", [6, 11, 13, 18])  # 128, 64, 96 and 192 rows
@pytest.mark.parametrize("n,k", [(64, 128), (320, 96), (256, 608)])  # an odd number of 64-byte steps; several periods
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_fragments(variant, n, k, act, dtype):
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(n + k)
    E, rows, n_out = len(ROWS), sum(ROWS), n // 2 if act else n
    # (a source row per sorted row, not its own: the rows are gathered)
    src = torch.randperm(rows, generator=gen)
    a = torch.randn(rows, k, generator=gen).to(dtype).cuda()
    w = (torch.randn(E, n, k, generator=gen) * 0.05).to(dtype).cuda()
    tiled = torch.empty_like(w)
    L.check(L.lib.kmoe_tile_weights_i8(w.data_ptr(), tiled.data_ptr(), E, n, 2 * k, L.stream()))
    lod = torch.tensor([0] + ROWS).cumsum(0).int().cuda()
    dsrc = src.int().cuda()
    y = torch.full((rows, n_out), float("nan"), dtype=dtype, device="cuda")
    g = L.GemmBf16Args()
    g.a, g.lda, g.row_src, g.src_div = a.data_ptr(), k, dsrc.data_ptr(), 1
    g.w, g.w_layout, g.lod = tiled.data_ptr(), L.KMOE_W_TILED, lod.data_ptr()
    g.E, g.n, g.k, g.rows = E, n, k, rows
    g.y, g.ldy, g.act, g.variant = y.data_ptr(), n_out, act, variant
    g.act_dtype = L.act_dtype(a, "test")
    L.check(L.lib.kmoe_grouped_gemm_bf16(g, L.stream()))
    ref = torch.cat([a[src[lo:lo + c]].float() @ w[e].float().T
                     for e, (c, lo) in enumerate(zip(ROWS, lod.tolist()))])
    if act:
        gate, up = (t.to(dtype).float() for t in ref.split(n_out, 1))
        ref = torch.nn.functional.silu(gate) * up
    got = y.float()
    assert not got.isnan().any()
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp(min=1e-6)
    assert float((got - ref).norm() / ref.norm()) <= 4e-3 and float(per_row.max()) <= 2e-2


@pytest.mark.parametrize("variant", [16, 32, 64, 96, 128])
@pytest.mark.parametrize("blocks", [1, 2, 3, 5])  # 128-value blocks: fewer than a turn of the rings, a turn, turns and a rest
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_packed_tiles_give_the_streaming_kernels_bits(variant, blocks, act, dtype):
    """4-bit weights: every tile height against the streaming kernel's launches that do not split K (variant 1), which
    add the same products in the same order, and both, with the launch the sizes choose (variant 0), against a float32
    product of the unpacked values."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(blocks)
    counts = ROWS + [31, 32, 63, 64, 65]
    E, rows, n, k, group = len(counts), sum(counts), 160, 128 * blocks, 32
    src = torch.randperm(rows, generator=gen).int().cuda()
    a = torch.randn(rows, k, generator=gen).to(dtype).cuda()
    packed = torch.randint(0, 256, (E, n, k // 2), generator=gen, dtype=torch.uint8).cuda()
    scale = (torch.rand(E, n, k // group, generator=gen) * 0.02 + 0.002).to(dtype).cuda()
    tiled = torch.empty_like(packed)
    L.check(L.lib.kmoe_tile_weights_i8(packed.data_ptr(), tiled.data_ptr(), E, n, k // 2, L.stream()))
    lod = torch.tensor([0] + counts).cumsum(0).int().cuda()
    n_out = n // 2 if act else n
    out = []
    for v in (1, variant, 0):
        y = torch.full((rows, n_out), float("nan"), dtype=dtype, device="cuda")
        g = L.GemmW4Args()
        g.a, g.lda, g.row_src, g.src_div = a.data_ptr(), k, src.data_ptr(), 1
        g.w, g.w_scale, g.group_size, g.lod = tiled.data_ptr(), scale.data_ptr(), group, lod.data_ptr()
        g.E, g.n, g.k, g.rows, g.w_layout = E, n, k, rows, L.KMOE_W_TILED
        g.y, g.ldy, g.act, g.variant, g.act_dtype = y.data_ptr(), n_out, act, v, L.act_dtype(a, "test")
        L.check(L.lib.kmoe_grouped_gemm_w4a16(g, L.stream()))
        out.append(y)
    assert not out[0].isnan().any() and torch.equal(out[0], out[1])
    ref = torch.cat([a[src[lo:lo + c].long()].float() @ _dequantised(packed[e], scale[e], dtype).T
                     for e, (c, lo) in enumerate(zip(counts, lod.tolist()))])
    if act:
        gate, up = (t.to(dtype).float() for t in ref.split(n_out, 1))
        ref = torch.nn.functional.silu(gate) * up
    for y in out[1:]:
        per_row = (y.float() - ref).norm(dim=1) / ref.norm(dim=1).clamp(min=1e-6)
        assert float((y.float() - ref).norm() / ref.norm()) <= 4e-3 and float(per_row.max()) <= 2e-2


def _dequantised(packed, scale, dtype):
    """[n, k/2] codes and [n, k/32] scales -> the values the kernels multiply, in float32."""
    codes = torch.stack([packed & 15, packed >> 4], -1).reshape(packed.shape[0], -1).float() - 8
    return (codes * scale.float().repeat_interleave(32, 1)).to(dtype).float()


@pytest.mark.parametrize("variant", [16, 32, 64, 96, 128])
@pytest.mark.parametrize("blocks,group", [(1, 32), (1, 128), (2, 256), (3, 64), (5, 32), (8, 1024), (9, 128), (9, 384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_packed_tiles_take_scales_by_chunks(variant, blocks, group, dtype):
    """Re-arranged group scales (which the tile kernel copies several blocks at a time: less than a chunk, chunks and a rest, groups of
    part of a block to several chunks) give the bits of row-major ones, and so do scales that begin between 16-byte boundaries."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(blocks + group)
    counts = [variant + 1, 0, 1, 17]
    E, rows, n, k = len(counts), sum(counts), 160, 128 * blocks
    groups = k // group
    a = torch.randn(rows, k, generator=gen).to(dtype).cuda()
    packed = torch.randint(0, 256, (E, n, k // 2), generator=gen, dtype=torch.uint8).cuda()
    scale = (torch.rand(E, n, groups, generator=gen) * 0.02 + 0.002).to(dtype).cuda()
    tiled, chunks = torch.empty_like(packed), torch.empty_like(scale)
    L.check(L.lib.kmoe_tile_weights_i8(packed.data_ptr(), tiled.data_ptr(), E, n, k // 2, L.stream()))
    L.check(L.lib.kmoe_tile_scales_w4(scale.data_ptr(), chunks.data_ptr(), E, n, groups, L.stream()))
    shifted = torch.empty(scale.numel() + 8, dtype=dtype, device="cuda")[4:-4].copy_(chunks.flatten())
    lod = torch.tensor([0] + counts).cumsum(0).int().cuda()
    for act in (0, 1):
        out, by_chunks = [], []
        for s, layout in ((scale, L.KMOE_S_ROWMAJOR), (chunks, L.KMOE_S_FRAG16), (shifted, L.KMOE_S_FRAG16)):
            y = torch.full((rows, n // 2 if act else n), float("nan"), dtype=dtype, device="cuda")
            g = L.GemmW4Args()
            g.a, g.lda, g.src_div, g.scale_layout = a.data_ptr(), k, 1, layout
            g.w, g.w_scale, g.group_size, g.lod = tiled.data_ptr(), s.data_ptr(), group, lod.data_ptr()
            g.E, g.n, g.k, g.rows, g.w_layout = E, n, k, rows, L.KMOE_W_TILED
            g.y, g.ldy, g.act, g.variant, g.act_dtype = y.data_ptr(), y.shape[1], act, variant, L.act_dtype(a, "test")
            L.lib.kmoe_trace_kernels(1)
            L.check(L.lib.kmoe_grouped_gemm_w4a16(g, L.stream()))
            by_chunks.append("scales by chunks" in L.lib.kmoe_traced_kernels().decode())
            L.lib.kmoe_trace_kernels(0)
            out.append(y)
        assert by_chunks == [False, group != 384, False]
        assert not out[0].isnan().any() and torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.parametrize("variant", [0, 1, 2, 4])
@pytest.mark.parametrize("act,gather", [(0, False), (1, False), (1, True)])
def test_packed_weights_on_rows_far_apart(variant, act, gather):
    """4-bit weights and activation rows 128 MiB apart: the last ones lie beyond 4 GiB, the reach of a 32-bit offset."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(variant + act)
    counts, n, k, lda = [9, 0, 20, 11], 64, 256, 1 << 26
    E, rows, n_out = len(counts), sum(counts), n // 2 if act else n
    a = torch.randn(rows, k, generator=gen).bfloat16().cuda()
    far = torch.empty(rows * lda, dtype=torch.bfloat16, device="cuda").view(rows, lda)
    far[:, :k] = a
    src = torch.randperm(rows, generator=gen) if gather else torch.arange(rows)
    dsrc = src.int().cuda()
    packed = torch.randint(0, 256, (E, n, k // 2), generator=gen, dtype=torch.uint8).cuda()
    scale = (torch.rand(E, n, k // 32, generator=gen) * 0.02 + 0.002).bfloat16().cuda()
    tiled = torch.empty_like(packed)
    L.check(L.lib.kmoe_tile_weights_i8(packed.data_ptr(), tiled.data_ptr(), E, n, k // 2, L.stream()))
    lod = torch.tensor([0] + counts).cumsum(0).int().cuda()
    y = torch.full((rows, n_out), float("nan"), dtype=torch.bfloat16, device="cuda")
    g = L.GemmW4Args()
    g.a, g.lda, g.row_src, g.src_div = far.data_ptr(), lda, dsrc.data_ptr() if gather else None, 1
    g.w, g.w_scale, g.group_size, g.lod = tiled.data_ptr(), scale.data_ptr(), 32, lod.data_ptr()
    g.E, g.n, g.k, g.rows, g.w_layout = E, n, k, rows, L.KMOE_W_TILED
    g.y, g.ldy, g.act, g.variant, g.act_dtype = y.data_ptr(), n_out, act, variant, L.KMOE_DT_BF16
    L.check(L.lib.kmoe_grouped_gemm_w4a16(g, L.stream()))
    ref = torch.cat([a[src[lo:lo + c]].float() @ _dequantised(packed[e], scale[e], torch.bfloat16).T
                     for e, (c, lo) in enumerate(zip(counts, lod.tolist()))])
    if act:
        gate, up = (t.bfloat16().float() for t in ref.split(n_out, 1))
        ref = torch.nn.functional.silu(gate) * up
    got = y.float()
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp(min=1e-6)
    assert not got.isnan().any() and float(per_row.max()) <= 2e-2


@pytest.mark.parametrize("variant", [0, 18, 19, 20])  # the height the sizes choose; 192, 128 and 160 rows
@pytest.mark.parametrize("blocks", [3, 4, 5, 9])  # row scales travel four blocks at a time: too few, one group, a rest
@pytest.mark.parametrize("act,dtype", [(0, torch.float16), (0, torch.bfloat16), (1, torch.bfloat16)])
@pytest.mark.parametrize("tail", [0, 161])
def test_block_fp8_wide_tiles(variant, blocks, act, dtype, tail):
    """fp8 with 128-wide block scales: the wide tiles at the edges of their heights, rows gathered, with and without a
    tail expert. The products are exact and summed in float32: what is left without SiLU is the rounding of the result,
    half a unit of bfloat16's eight bits (2**-8). With it, a gate or up value whose float32 sums lie on both sides of a tie is rounded to
    neighbours, a whole unit (2 * 2**-8) for each of the two; one large value can carry a row of 128 results."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(100 * blocks + tail)
    counts = ROWS + [159, 160, 161, 319, 321, 384, 385]
    E, rows, n, k = len(counts), sum(counts), 384 - 128 * act, 128 * blocks
    n_out = n // 2 if act else n
    fp8 = torch.float8_e4m3fn
    a = torch.randn(rows + tail, k, generator=gen).to(fp8).cuda()
    a_scale = (torch.rand(rows + tail, blocks, generator=gen) + 0.5).cuda()
    w = torch.randn(E + 1, n, k, generator=gen).to(fp8).cuda()
    w_scale = (torch.rand(E + 1, n // 128, blocks, generator=gen) + 0.5).cuda()
    tiled = torch.empty_like(w)
    L.check(L.lib.kmoe_tile_weights_i8(w.data_ptr(), tiled.data_ptr(), E + 1, n, k, L.stream()))
    src = torch.randperm(rows, generator=gen).cuda()
    dsrc, lod = src.int(), torch.tensor([0] + counts).cumsum(0).int().cuda()
    y = torch.full((rows + tail, n_out), float("nan"), dtype=dtype, device="cuda")
    g = L.GemmFp8Args()
    g.a, g.lda, g.a_scale, g.row_src, g.src_div = a.data_ptr(), k, a_scale.data_ptr(), dsrc.data_ptr(), 1
    g.w, g.w_scale, g.w_layout, g.lod = tiled.data_ptr(), w_scale.data_ptr(), L.KMOE_W_TILED, lod.data_ptr()
    g.E, g.n, g.k, g.rows = E, n, k, rows
    g.y, g.ldy, g.act, g.variant, g.act_dtype = y.data_ptr(), n_out, act, variant, L.act_dtype(y, "test")
    if tail:
        g.w_tail, g.w_scale_tail = tiled[E].data_ptr(), w_scale[E].data_ptr()
        g.tail_row0, g.tail_rows, g.tail_src0 = rows, tail, rows
    L.check(L.lib.kmoe_grouped_gemm_fp8_block(g, L.stream()))
    a_full = a.float() * a_scale.repeat_interleave(128, 1)
    w_full = w.float() * w_scale.repeat_interleave(128, 1).repeat_interleave(128, 2)
    parts = [a_full[src[lo:lo + c]] @ w_full[e].T for e, (c, lo) in enumerate(zip(counts, lod.tolist()))]
    ref = torch.cat(parts + [a_full[rows:] @ w_full[E].T])
    if act:
        gate, up = (t.to(dtype).float() for t in ref.split(n_out, 1))
        ref = torch.nn.functional.silu(gate) * up
    got = y.float()
    assert not got.isnan().any()
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp(min=1e-6)
    assert float(per_row.max()) <= (5 if act else 1) * 2 ** -8


@pytest.mark.parametrize("variant,rows", [(19, 128), (20, 160), (18, 192)])
@pytest.mark.parametrize("blocks", [3, 4])
def test_block_fp8_wide_tiles_need_four_blocks(variant, rows, blocks):
    """A forced wide tile runs from four blocks of K on; with fewer the launch is the four-wave tiles'. The bits are the same."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator().manual_seed(blocks)
    counts = [200, 0, 17]
    E, n, k, fp8 = len(counts), 256, 128 * blocks, torch.float8_e4m3fn
    a = torch.randn(sum(counts), k, generator=gen).to(fp8).cuda()
    a_scale = (torch.rand(sum(counts), blocks, generator=gen) + 0.5).cuda()
    w = torch.randn(E, n, k, generator=gen).to(fp8).cuda()
    w_scale = (torch.rand(E, n // 128, blocks, generator=gen) + 0.5).cuda()
    lod = torch.tensor([0] + counts).cumsum(0).int().cuda()
    out = []
    for v in (variant, 6):
        y = torch.zeros(sum(counts), n, dtype=torch.bfloat16, device="cuda")
        g = L.GemmFp8Args()
        g.a, g.lda, g.a_scale, g.src_div, g.w, g.w_scale = a.data_ptr(), k, a_scale.data_ptr(), 1, w.data_ptr(), w_scale.data_ptr()
        g.w_layout, g.lod, g.E, g.n, g.k, g.rows = L.KMOE_W_TILED, lod.data_ptr(), E, n, k, sum(counts)
        g.y, g.ldy, g.variant, g.act_dtype = y.data_ptr(), n, v, L.act_dtype(y, "test")
        L.lib.kmoe_trace_kernels(1)
        L.check(L.lib.kmoe_grouped_gemm_fp8_block(g, L.stream()))
        L.lib.kmoe_trace_kernels(0)
        out.append((y, L.lib.kmoe_traced_kernels().decode()))
    assert f"{rows if blocks >= 4 else 128}x256 tile, {8 if blocks >= 4 else 4} waves" in out[0][1], out[0][1]
    assert "128x256 tile, 4 waves" in out[1][1], out[1][1]
    assert torch.equal(out[0][0], out[1][0])


@pytest.mark.parametrize("fmt", ["int8", "fp8"])
@pytest.mark.parametrize("counts", [[64, 1, 65, 130] * 16, [3, 0, 129, 640, 64], [1, 63], [40], [200]],
                         ids=lambda c: "-".join(map(str, c[:5])))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", [False, True])
@pytest.mark.parametrize("k", [384, 640, 1024])  # whole and partial periods of the loop
def test_64_row_tiles_read_what_one_tile_reads_past_the_caches(fmt, counts, dtype, act, k):
    """Experts with one tile and with several in a launch, one after the other on the same workgroup too; one matrix alone. The
    bits are the 128-row tiles'."""
    from vllm_kunlun_amd import _lib as L
    gen = torch.Generator(device="cuda").manual_seed(sum(counts))
    E, n, rows = len(counts), 2048, sum(counts)
    lod = torch.tensor([0] + counts).cumsum(0).int().cuda()
    if fmt == "int8":
        g, call = L.GemmI8Args(), L.lib.kmoe_grouped_gemm_i8
        a, w = (torch.randint(-127, 128, shape, generator=gen, dtype=torch.int8, device="cuda") for shape in ((rows, k), (E, n, k)))
        scales = [torch.rand(shape, generator=gen, device="cuda") + 0.5 for shape in ((rows,), (E, n))]
        g.a_max, g.w_max = (t.data_ptr() for t in scales)
    else:
        g, call = L.GemmFp8Args(), L.lib.kmoe_grouped_gemm_fp8_block
        a, w = (torch.randn(shape, generator=gen, device="cuda").to(torch.float8_e4m3fn) for shape in ((rows, k), (E, n, k)))
        scales = [torch.rand(shape, generator=gen, device="cuda") + 0.5 for shape in ((rows, k // 128), (E, n // 128, k // 128))]
        g.a_scale, g.w_scale = (t.data_ptr() for t in scales)
    g.a, g.lda, g.src_div, g.w, g.w_layout, g.lod = a.data_ptr(), k, 1, w.data_ptr(), L.KMOE_W_TILED, lod.data_ptr()
    g.E, g.n, g.k, g.rows, g.act = E, n, k, rows, L.KMOE_ACT_SWIGLU if act else L.KMOE_ACT_NONE
    out = []
    for variant in (11, 6):
        y = torch.zeros(rows, n // 2 if act else n, dtype=dtype, device="cuda")
        g.y, g.ldy, g.variant, g.act_dtype = y.data_ptr(), y.shape[1], variant, L.act_dtype(y, "test")
        L.lib.kmoe_trace_kernels(1)
        L.check(call(g, L.stream()))
        L.lib.kmoe_trace_kernels(0)
        out.append((y, L.lib.kmoe_traced_kernels().decode()))
    assert "64x256 tile" in out[0][1] and ("weights past the caches" in out[0][1]) == (E > 1), out[0][1]
    assert "128x256 tile" in out[1][1] and torch.equal(out[0][0], out[1][0])
