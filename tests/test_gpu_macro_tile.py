"""The tiles with both operands in LDS (variant 23) against the 128-row tiles (variant 6; fp8: the 128-row wide tiles, 19), which add
the same products in the same order: the same bits, at the edges of row fragments and tiles, of the channels, for every form of the
operands' rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FEW = [0, 1, 2, 0, 3] * 12  # with these an expert holds few rows on average: the lower tiles of fp8
ROWS = [1, 15, 16, 17, 0, 191, 192, 193, 33, 384, 385, 0, 127, 128, 129, 800, 3100]  # up to 17 tiles of an expert


def _launch(kind, counts, n, k, act, dtype, div=1, gather=True, pad=0, tail=0, bound=0, seed=0, variant=23, trace=False, strange=False, reference=False):
    """Outputs of the variants 6 and 23 (or another) for the same operands; trace: and the latter's kernel. pad: values between the rows of a and y; tail: rows of an expert
    outside w (int8); bound: rows the caller allows for beyond the last expert's; strange: infinities and NaN in some rows of a;
    reference: the second is the float32 product of the dequantised operands instead."""
    from vllm_kunlun_amd import _lib as L
    g = torch.Generator(device="cuda").manual_seed(seed)
    E, rows, n_out = len(counts), sum(counts), n // 2 if act else n
    a_rows = (-(-rows // div) if gather else rows) + tail
    src = torch.randperm(rows, generator=g, device="cuda").int()
    lod = torch.tensor([0] + counts).cumsum(0).int().cuda()
    i8, f8 = kind == "int8", kind == "fp8"
    if f8:
        a, w = (torch.randn(shape, generator=g, device="cuda").mul_(60).to(torch.float8_e4m3fn) for shape in ((a_rows, k + pad), (E + 1, n, k)))
        a_max, w_max = (torch.rand(shape, generator=g, device="cuda") * 0.01 + 0.001 for shape in ((a_rows, k // 128), (E + 1, n // 128, k // 128)))
    else:
        a_max, w_max = (torch.rand(shape, generator=g, device="cuda") * 0.1 + 0.01 for shape in ((a_rows,), (E + 1, n)))
    if not f8:
        a = (torch.randint(-127, 128, (a_rows, k + pad), generator=g, device="cuda", dtype=torch.int8) if i8
             else torch.randn(a_rows, k + pad, generator=g, device="cuda").to(dtype))
        w = (torch.randint(-127, 128, (E + 1, n, k), generator=g, device="cuda", dtype=torch.int8) if i8
             else torch.randn(E + 1, n, k, generator=g, device="cuda").mul_(0.05).to(dtype))
    if strange and f8:
        a[5:200:40].view(torch.int8)[:, 3] = 0x7f  # NaN
        a_max[7:200:40, 1] = float("inf")
    elif strange:
        a[5:200:40, 3], a[7:200:40, 700] = float("nan"), float("inf")
    tiled = torch.empty_like(w)
    L.check(L.lib.kmoe_tile_weights_i8(w.data_ptr(), tiled.data_ptr(), E + 1, n, k * w.element_size(), L.stream()))
    q = L.GemmI8Args() if i8 else (L.GemmFp8Args() if f8 else L.GemmBf16Args())
    if i8 or f8:
        for name, scales in (("a_max", a_max), ("w_max", w_max)) if i8 else (("a_scale", a_max), ("w_scale", w_max)):
            setattr(q, name, scales.data_ptr())
        if tail:
            q.w_tail = tiled[E].data_ptr()
            setattr(q, "w_max_tail" if i8 else "w_scale_tail", w_max[E].data_ptr())
            q.tail_row0, q.tail_rows, q.tail_src0 = rows, tail, a_rows - tail
    q.a, q.lda, q.w, q.w_layout, q.lod = a.data_ptr(), k + pad, tiled.data_ptr(), L.KMOE_W_TILED, lod.data_ptr()
    q.row_src, q.src_div = (src.data_ptr(), div) if gather else (0, 1)
    q.E, q.n, q.k, q.rows, q.act, q.ldy = E, n, k, rows + bound, act, n_out + pad
    out = []
    for v in (19 if f8 else 6, variant):
        y = torch.full((rows + tail, n_out + pad), float("nan"), dtype=dtype, device="cuda")
        q.y, q.variant, q.act_dtype = y.data_ptr(), v, L.act_dtype(y, "test")
        launch = L.lib.kmoe_grouped_gemm_i8 if i8 else (L.lib.kmoe_grouped_gemm_fp8_block if f8 else L.lib.kmoe_grouped_gemm_bf16)
        L.lib.kmoe_trace_kernels(1)
        L.check(launch(q, L.stream()))
        L.lib.kmoe_trace_kernels(0)
        out.append(y)
    torch.cuda.synchronize()
    if reference:
        rows_of_a = (src.long() // div if gather else torch.arange(rows, device="cuda"))
        x = a[:, :k].float()
        x = x * (a_max.repeat_interleave(128, 1) if f8 else (a_max / 127)[:, None]) if i8 or f8 else x
        for e in range(E):
            if counts[e]:
                we = w[e].float()
                we = we * (w_max[e].repeat_interleave(128, 0).repeat_interleave(128, 1) if f8 else (w_max[e] / 127)[:, None]) if i8 or f8 else we
                at = slice(int(lod[e]), int(lod[e + 1]))
                v = x[rows_of_a[at]] @ we.t()
                if act:
                    gate, up = (t.to(dtype).float() for t in v.split(n_out, 1))
                    v = torch.nn.functional.silu(gate) * up
                out[0][at, :n_out] = v.to(dtype)
    return (out, n_out, L.lib.kmoe_traced_kernels().decode()) if trace else (out, n_out)


def _same(out, n_out):
    assert not out[1][:, :n_out].isnan().any() and torch.equal(out[0][:, :n_out], out[1][:, :n_out])
    assert out[1][:, n_out:].isnan().all()  # nothing between the rows is written


@pytest.mark.parametrize("kind", ["int8", "16 bit"])
@pytest.mark.parametrize("n,k", [(64, 768), (320, 896), (256, 1024), (544, 2048)])  # bytes of K: 12, 14, 16, 32 steps
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tiles(kind, n, k, act, dtype):
    _same(*_launch(kind, ROWS, n, k if kind == "int8" else k // 2, act, dtype, div=8))


@pytest.mark.parametrize("kind", ["int8", "16 bit", "fp8"])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_float32(kind, act, dtype):
    """The bounds that the other tiles are held to against the product of the same values in float32: two roundings of 2^-9 relative
    (gate and up before SiLU-mul, and the result)."""
    out, n_out = _launch(kind, ROWS, 512, 768, act, dtype, div=8, reference=True)
    ref, got = (o[:, :n_out].float() for o in out)
    assert not got.isnan().any()
    per_row = (got - ref).norm(dim=1) / ref.norm(dim=1).clamp(min=1e-6)
    assert float((got - ref).norm() / ref.norm()) <= 4e-3 and float(per_row.max()) <= 2e-2


@pytest.mark.parametrize("n,k", [(256, 768), (768, 896), (512, 1024), (512, 1152), (256, 2048)])  # 6 to 9 and 16 blocks of K
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("few", [False, True])
def test_tiles_fp8(n, k, act, dtype, few):
    _same(*_launch("fp8", [r for r in ROWS if r < 800] + FEW if few else ROWS, n, k, act, dtype, div=8))


def test_channels_that_end_inside_a_tile_fp8():
    _same(*_launch("fp8", ROWS, 384, 896, 0, torch.bfloat16))


@pytest.mark.parametrize("kind", ["int8", "16 bit", "fp8"])
@pytest.mark.parametrize("form", [dict(gather=False), dict(div=1), dict(div=3), dict(div=6), dict(pad=64), dict(bound=500)], ids=str)
@pytest.mark.parametrize("act", [0, 1])
def test_forms(kind, form, act):
    _same(*_launch(kind, ROWS, 512 if kind == "fp8" else 288, 768, act, torch.bfloat16, **form))


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("tail", [1, 192, 700])
@pytest.mark.parametrize("act", [0, 1])
def test_tail_expert(kind, tail, act):
    _same(*_launch(kind, ROWS, 512 if kind == "fp8" else 288, 768, act, torch.bfloat16, div=8, tail=tail))


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("counts", [[], [1], [193], [5] * 40], ids=len)  # routed items: none, fewer than XCDs, of two tiles, some each
@pytest.mark.parametrize("tail", [7, 1600, 3100])
def test_tail_expert_beside_few_items(kind, counts, tail):
    counts = counts or [0]
    _same(*_launch(kind, counts, 1024, 768, 0, torch.bfloat16, tail=tail))


def test_more_items_than_are_resolved_at_once():
    """Over 32 items per workgroup, and weights beyond the memory-side cache: those of experts with one tile are read past it."""
    _same(*_launch("int8", [1, 192, 193, 0, 40] * 28, 16384, 768, 0, torch.bfloat16))


@pytest.mark.parametrize("kind,k,div,experts", [("int8", 640, 1, 3), ("int8", 832, 1, 3), ("int8", 768, 5, 3), ("int8", 768, 1, 500), ("16 bit", 352, 1, 3), ("16 bit", 416, 1, 3),
                                                ("16 bit", 384, 5, 3), ("16 bit", 384, 1, 500), ("fp8", 640, 1, 3), ("fp8", 768, 5, 3), ("fp8", 768, 1, 500)])
def test_what_the_launch_does_not_take(kind, k, div, experts):
    """Too short a K, no whole chunks, a divisor whose quotients one multiplication does not give, too many experts for its LDS:
    refused when asked for by name."""
    with pytest.raises(NotImplementedError, match="variant 23 needs"):
        _launch(kind, [5] * experts, 128, k, 0, torch.bfloat16, div=div)


@pytest.mark.parametrize("kind,E,n,k,act,rows,div,tile", [
    ("int8", 96, 2560, 2048, 1, 100, 6, True), ("int8", 96, 2560, 2048, 1, 100, 5, False), ("int8", 96, 2560, 1984, 1, 100, 1, False),
    ("int8", 411, 1024, 2048, 1, 20, 1, True), ("int8", 412, 1024, 2048, 1, 20, 1, False),
    ("16 bit", 96, 3072, 1024, 0, 100, 6, True), ("16 bit", 96, 3072, 1024, 0, 100, 5, False), ("16 bit", 96, 3072, 1056, 0, 100, 1, False), ("16 bit", 412, 1024, 512, 0, 15, 1, False),
    ("fp8", 96, 3072, 2048, 1, 150, 6, True), ("fp8", 96, 3072, 2048, 1, 150, 5, False), ("fp8", 412, 1024, 2048, 1, 20, 1, False)])
def test_served_by_another_kernel(kind, E, n, k, act, rows, div, tile):
    """Launches that the choice would give to the tile and whose form it does not take, beside their neighbours that it does."""
    out, n_out, ran = _launch(kind, [rows] * E, n, k, act, torch.bfloat16, div=div, variant=0, trace=True)
    _same(out, n_out)
    assert ("both operands" in ran) == tile, ran


def test_accumulators_are_served_by_another_kernel():
    """int32 accumulators (asymmetric activations) of a matrix whose plain product takes the tile."""
    from vllm_kunlun_amd import _lib as L
    from vllm_kunlun_amd.ops import _custom_ops  # noqa: F401
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randint(-127, 128, (3500, 768), generator=g, device="cuda", dtype=torch.int8)
    w = torch.randint(-127, 128, (12288, 768), generator=g, device="cuda", dtype=torch.int8)
    one = torch.ones(1, 1, device="cuda")
    from vllm_kunlun_amd._plan import tile_int8_weights_
    want = a.float() @ w.float().t()  # (sums below 2^24: exact)
    tile_int8_weights_(w)
    L.lib.kmoe_trace_kernels(1)
    got = torch.ops._C.cutlass_scaled_mm_azp(a, w.t(), one, one, torch.bfloat16, torch.zeros(1, 12288, dtype=torch.int32, device="cuda"))
    L.lib.kmoe_trace_kernels(0)
    ran = L.lib.kmoe_traced_kernels().decode()
    assert "tiled_gemm_kernel" in ran and "both operands" not in ran, ran
    assert torch.equal(got, want.bfloat16())


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("few", [False, True])
def test_longest_k_fp8(act, few):
    """64 blocks of K: the most whose weight scales its LDS holds."""
    _same(*_launch("fp8", [r for r in ROWS if r < 400] + FEW if few else ROWS, 256, 8192, act, torch.bfloat16, div=8))


@pytest.mark.parametrize("kind", ["16 bit", "fp8"])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinities_and_nan_stay_in_their_rows(kind, act, dtype):
    """Operand rows of infinities and of NaN (fp8: its NaN; its scales infinite): those rows as the other kernel has them, all others
    their own values, and results beyond the largest half or bfloat16."""
    out, n_out = _launch(kind, ROWS, 512, 768, act, dtype, strange=True)
    a, b = (o[:, :n_out].float() for o in out)
    assert a.isnan().any() and a.isinf().any() and a.isfinite().any(dim=1).any()
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("n,k,rows,tile", [
    (7168, 768, 700, "64x256 tile, 4 waves"), (7168, 768, 1400, "192x256 tile, 8 waves"), (7168, 640, 1400, "192x256 tile, 8 waves"),
    (12288, 768, 3500, "192x256 tile, both"), (7168, 4096, 1900, "128x256 tile, 4 waves"), (4096, 4096, 4000, "128x256 tile, 4 waves"),
    # channel blocks for every CU: by the rows alone
    (65536, 128, 64, "64x256 tile, 4 waves"), (65536, 128, 65, "96x256 tile, 4 waves"), (65536, 128, 96, "96x256 tile, 4 waves"),
    (65536, 128, 97, "128x256 tile, 8 waves"), (65536, 128, 129, "192x256 tile, 8 waves"), (65536, 128, 193, "128x256 tile, 4 waves"),
    (65536, 128, 257, "192x256 tile, 8 waves"), (65536, 4096, 300, "192x256 tile, 8 waves")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_matrix_alone(n, k, rows, tile, dtype):
    """The tile for one matrix: by rounds of workgroups, by the rows where one row of tiles fills every CU, and the macro tile over short K."""
    out, n_out, ran = _launch("int8", [rows], n, k, 0, dtype, gather=False, variant=0, trace=True)
    _same(out, n_out)
    assert tile in ran, ran


@pytest.mark.parametrize("n,k,rows,experts", [(7168, 768, 300, 4), (1536, 768, 150, 32), (1536, 768, 300, 16), (512, 4096, 150, 128), (512, 4096, 400, 128)])
def test_less_than_a_round(n, k, rows, experts):
    """Few tiles for the CUs, and a long K."""
    _same(*_launch("int8", [rows] * experts, n, k, 0, torch.bfloat16, variant=0))


MACRO, LOW = "192x256 tile, both", "128x256 tile, both"


def _runs(kind, E, n, k, act, rows, tile):
    """The launch of E experts of `rows` rows each gives the 128-row tile's bits; `tile`: part of its kernel's name, or None for any but the macro tile."""
    out, n_out, ran = _launch(kind, [rows] * E, n, k, act, torch.bfloat16, gather=False, variant=0, trace=True)
    _same(out, n_out)
    assert (tile in ran) if tile else ("both operands" not in ran), ran


@pytest.mark.parametrize("E,n,k,act,rows,tile", [
    (64, 1024, 1024, 1, 111, None), (64, 1024, 1024, 1, 384, None), (64, 1024, 1024, 1, 385, MACRO), (96, 2048, 1024, 1, 100, None), (96, 2048, 1024, 1, 111, MACRO),
    (64, 2304, 2048, 1, 105, None), (64, 2304, 2048, 1, 123, None), (64, 2304, 2048, 1, 124, MACRO), (64, 2304, 2048, 1, 176, None), (32, 2304, 2048, 1, 900, None),
    (96, 3072, 2048, 0, 105, LOW), (96, 3072, 2048, 0, 111, None), (96, 3072, 2048, 0, 300, None), (96, 3072, 2048, 0, 301, MACRO), (96, 2816, 768, 0, 100, None)])
def test_choice_fp8(E, n, k, act, rows, tile):
    """Experts an XCD's L2 holds and larger ones, in fewer rounds and more, one tile and several; a launch whose weights the memory-side cache holds."""
    _runs("fp8", E, n, k, act, rows, tile)


@pytest.mark.parametrize("E,n,k,act,rows,tile", [
    (80, 2304, 1024, 0, 18, MACRO), (80, 2304, 1024, 0, 19, None), (80, 2304, 1024, 0, 27, None), (80, 2304, 1024, 0, 28, MACRO),
    (80, 2304, 1024, 0, 172, MACRO), (80, 2304, 1024, 0, 173, None), (80, 2304, 1024, 0, 280, None), (80, 2304, 1024, 0, 281, MACRO),
    (128, 2048, 768, 0, 200, MACRO), (64, 2304, 2048, 0, 400, MACRO), (64, 2304, 2048, 0, 401, None), (1, 65536, 2048, 0, 200, None),
    (1, 131072, 1152, 0, 160, None), (1, 131072, 1152, 0, 161, MACRO),
    (64, 4096, 1024, 1, 72, None), (64, 4096, 1024, 1, 73, MACRO), (64, 4096, 1024, 1, 163, MACRO), (64, 4096, 1024, 1, 170, None)])
def test_choice_16_bit(E, n, k, act, rows, tile):
    """Few rows, one tile, the beginning of a second, a long K, one matrix; gate_up."""
    _runs("16 bit", E, n, k, act, rows, tile)


@pytest.mark.parametrize("E,n,k,act,rows,tile", [
    (96, 3072, 2048, 1, 60, MACRO), (96, 2560, 2048, 1, 72, None), (96, 2560, 2048, 1, 73, MACRO), (64, 1024, 1024, 1, 193, None), (64, 1024, 1024, 1, 384, None),
    (64, 2048, 1024, 1, 193, MACRO), (64, 1024, 1024, 1, 385, MACRO), (128, 1024, 4096, 0, 88, None), (128, 1024, 4096, 0, 89, MACRO),
    (128, 1024, 4096, 0, 176, MACRO), (128, 1024, 4096, 0, 177, None), (16, 2048, 768, 0, 600, None), (16, 2048, 768, 0, 961, MACRO), (96, 2048, 768, 0, 88, None), (96, 2048, 768, 0, 89, MACRO)])
def test_choice_int8(E, n, k, act, rows, tile):
    """Four rounds and two, the second tile in few rounds, a long K, down launches in few rounds and more."""
    _runs("int8", E, n, k, act, rows, tile)


@pytest.mark.parametrize("fmt", ["int8", "fp8"])
@pytest.mark.parametrize("I,K,E,takes", [(768, 4, 16, True), (768, 6, 16, True), (640, 4, 16, False), (768, 5, 16, False), (768, 4, 416, False)])
def test_layer_asked_for_the_tile(fmt, I, K, E, takes):
    """tile_variant = 23 reaches both routed GEMMs where their shapes are what the tile takes, and is ignored otherwise."""
    from vllm_kunlun_amd import _lib as L
    from vllm_kunlun_amd import synth
    from vllm_kunlun_amd._plan import make_moe_plan
    shape = synth.scaled(synth.SHAPES["qwen3-decode"], M=300 * E // 16, H=1024, E=E, K=K, I=I)
    sl = (synth.make_w8a8_layer if fmt == "int8" else synth.make_fp8_layer)(shape, "cuda", seed=5)
    lay, outs = sl.layer, []
    for variant in (6 if fmt == "int8" else 19, 23):
        out = torch.empty_like(sl.x)
        plan = make_moe_plan(L.KMOE_FMT_INT8 if fmt == "int8" else L.KMOE_FMT_FP8_BLOCK, sl.x, sl.logits, out, shape.K, lay.w13_weight, lay.w2_weight,
                             lay.w13_weight_scale, lay.w2_weight_scale, shape.scoring, True, shape.n_group, shape.topk_group, 1.0, sl.bias, None, 1.0,
                             tile_variant=variant)
        L.lib.kmoe_trace_kernels(1)
        plan()
        L.lib.kmoe_trace_kernels(0)
        outs.append(out)
    torch.cuda.synchronize()
    ran = L.lib.kmoe_traced_kernels().decode()
    assert ran.count("both operands") == (2 if takes else 0), ran
    assert torch.equal(*outs)
