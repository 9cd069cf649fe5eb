"""Grouped expert GEMM (matrix cores) against an f32 torch reference of the same product.

The summation order differs from torch's, so the comparison is a tolerance, stated here:
|got - want| <= 1e-2 * |want| + 1e-2 * rms(want) (one bf16 ulp is 0.4-0.8 %; fp16 is tighter).
"""
import pytest
import torch

from kernel_amd import _lib
from kernel_amd import contract as C
from kernel_amd.all2all import HipAllToAll, concat_world
from oracle import all2all_vec as V

pytestmark = pytest.mark.gpu


def close(got, want):
    got, want = got.float().cpu(), want.float()
    tol = 1e-2 * want.abs() + 1e-2 * want.pow(2).mean().sqrt()
    bad = (got - want).abs() > tol
    assert not bool(bad.any()), f"{int(bad.sum())} of {bad.numel()} out of tolerance, worst " \
                                f"{float(((got - want).abs() / tol).max()):.2f}x"


def make(E, K, T, H, N, W, dtype, seed, zipf=False):
    g = torch.Generator().manual_seed(seed)
    cfg = C.MoEConfig(E, K, H, T + 1, dtype, dtype)
    if zipf:
        p = (torch.arange(E, dtype=torch.float64) + 1).pow(-1.2)
        idx = torch.multinomial((p / p.sum()).float().expand(T, E), K, generator=g).to(torch.int32)
    else:
        idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).to(torch.int32)
    world = [C.RankData(T, idx, torch.rand(T, K, generator=g), torch.randn(T, H, generator=g).to(dtype))]
    world += [C.RankData.empty(cfg) for _ in range(W - 1)]
    weights = (torch.randn(E, N, H, generator=g) / H ** 0.5).to(dtype)
    return cfg, world, weights


@pytest.mark.parametrize("E,K,T,H,N,W,zipf", [
    (8, 2, 40, 64, 64, 1, False),      # one K slab, tiles mostly empty
    (8, 2, 700, 128, 200, 2, False),   # several m-tiles per expert, N not a multiple of 128
    (16, 4, 300, 192, 136, 4, True),   # skewed: empty experts and long segments
    (64, 6, 1024, 2048, 2048, 8, True),
    (256, 8, 256, 7168, 512, 8, False),  # headline routing shape, 8 rows per expert on average
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("padded", [False, True], ids=["compact", "padded"])
@pytest.mark.parametrize("tile", ["32", "128", "256"], ids=["tile32", "tile128", "tile256"])
def test_expert_gemm_matches_f32_reference(gpu_device, options, E, K, T, H, N, W, zipf, dtype, padded, tile):
    # every kernel on every shape (the 32-row kernel needs H % 128 == 0; the library takes the
    # 128 x 128 kernel for the other hidden sizes)
    options.set("GEMM_TILE", tile)
    cfg, world, weights = make(E, K, T, H, N, W, dtype, seed=E + T, zipf=zipf)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, W, padded=padded, max_recv=T if padded else None)
    d = ata.dispatch(x, idx, rs)
    y = ata.expert_gemm(d, weights.to(gpu_device))
    torch.cuda.synchronize()
    o = V.run_world(cfg, world)
    want = V.expert_gemm(o["disp_x"], o["offsets"], weights, dtype)
    rows = d.slot_of_entry.long() if padded else o["slot_of_entry"].long().to(gpu_device)
    close(y[rows], want[o["slot_of_entry"].long()])
    if not padded:
        close(y, want)


@pytest.mark.parametrize("E,K,T,H,N,zipf", [
    (8, 2, 1200, 384, 264, False),   # 300 rows per expert: the library itself picks the 256 x 256 kernel
    (16, 4, 1500, 256, 512, True),   # skewed, segments from empty to well past one tile
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_both_tile_sizes_give_the_same_bits(gpu_device, options, E, K, T, H, N, zipf, dtype):
    """The two kernels accumulate over K in the same order, so their outputs are identical; the
    default choice for these shapes (R > 32 E) is the wide one."""
    cfg, world, weights = make(E, K, T, H, N, 1, dtype, seed=7 * E + T, zipf=zipf)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1)
    d = ata.dispatch(x, idx, rs)
    wd = weights.to(gpu_device)
    lib = ata.lib
    outs = {}
    for tile in ("default", "32", "128", "256"):
        if tile == "default":
            options.set("GEMM_TILE", 0)
        else:
            options.set("GEMM_TILE", tile)
        assert lib.moe_a2a_timer_begin(4) == 0
        outs[tile] = ata.expert_gemm(d, wd).clone()
        torch.cuda.synchronize()
        import ctypes
        ids, us = (ctypes.c_int * 4)(), (ctypes.c_float * 4)()
        assert lib.moe_a2a_timer_end(ids, us, 4) == 1
        name = lib.moe_a2a_kernel_name(ids[0]).decode()
        assert name == {"32": "expert_gemm_skinny", "128": "expert_gemm"}.get(tile, "expert_gemm_wide")
    assert torch.equal(outs["128"].view(torch.int16), outs["256"].view(torch.int16))
    assert torch.equal(outs["32"].view(torch.int16), outs["256"].view(torch.int16))
    assert torch.equal(outs["default"].view(torch.int16), outs["256"].view(torch.int16))
    o = V.run_world(cfg, world)
    close(outs["256"], V.expert_gemm(o["disp_x"], o["offsets"], weights, dtype))


@pytest.mark.parametrize("E,K,T,H,N,W,zipf", [
    (8, 2, 40, 128, 64, 1, False),      # one scale block, tiles mostly empty
    (8, 2, 1200, 256, 264, 2, False),   # full 256-row tiles and 128-row tails, ragged N
    (16, 4, 300, 384, 136, 4, True),    # skewed: empty experts and long segments
    (32, 4, 2048, 1024, 512, 8, False),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("padded", [False, True], ids=["compact", "padded"])
def test_expert_gemm_on_fp8_rows(gpu_device, E, K, T, H, N, W, zipf, dtype, padded):
    """fp8 dispatch -> expert GEMM.  The dispatched bytes and scales are bit-exact (checked here
    again), and the product is compared with an f32 matmul of the dequantised rows, each element
    rounded once to the weights' type as the kernel does."""
    cfg, world, weights = make(E, K, T, H, N, W, dtype, seed=3 * E + T, zipf=zipf)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, W, fp8_dispatch=True, padded=padded, max_recv=T if padded else None)
    d = ata.dispatch(x, idx, rs)
    y = ata.expert_gemm(d, weights.to(gpu_device))
    torch.cuda.synchronize()
    o = V.run_world(cfg, world, fp8=True)
    rows = d.slot_of_entry.long() if padded else o["slot_of_entry"].long().to(gpu_device)
    soe = o["slot_of_entry"].long()
    assert torch.equal(d.disp_x[rows].cpu(), o["disp_x"][soe])
    assert torch.equal(d.disp_scale[rows].cpu(), o["disp_scale"][soe])
    want = V.expert_gemm_fp8(o["disp_x"], o["disp_scale"], o["offsets"], weights, dtype)
    close(y[rows], want[soe])


def test_fp8_gemm_feeds_combine(gpu_device):
    """fp8 dispatch -> expert GEMM (H -> H) -> f32 combine against the same chain on the CPU."""
    cfg, world, weights = make(32, 4, 1024, 256, 256, 8, torch.bfloat16, seed=5)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 8, fp8_dispatch=True, combine_mode=C.COMBINE_F32)
    d = ata.dispatch(x, idx, rs)
    y = ata.combine(None, w, d, ata.expert_gemm(d, weights.to(gpu_device)))
    o = V.run_world(cfg, world, fp8=True)
    ey = V.expert_gemm_fp8(o["disp_x"], o["disp_scale"], o["offsets"], weights, torch.bfloat16)
    want = V.combine_f32(ey, w.cpu(), o["slot_of_entry"], torch.bfloat16)
    close(y, want)


def test_decode_shape_takes_the_skinny_kernel(gpu_device, options):
    """Eight rows per expert on average (the headline routing shape): the library picks the
    32 x 256 kernel by itself, and its bits equal the 128 x 128 kernel's."""
    options.set("GEMM_TILE", 0)
    cfg, world, weights = make(256, 8, 256, 1024, 520, 8, torch.bfloat16, seed=11)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 8)
    d = ata.dispatch(x, idx, rs)
    wd = weights.to(gpu_device)
    import ctypes
    assert ata.lib.moe_a2a_timer_begin(4) == 0
    y = ata.expert_gemm(d, wd).clone()
    torch.cuda.synchronize()
    ids, us = (ctypes.c_int * 4)(), (ctypes.c_float * 4)()
    assert ata.lib.moe_a2a_timer_end(ids, us, 4) == 1
    assert ata.lib.moe_a2a_kernel_name(ids[0]) == b"expert_gemm_skinny"
    options.set("GEMM_TILE", "128")
    y128 = ata.expert_gemm(d, wd)
    assert torch.equal(y.view(torch.int16), y128.view(torch.int16))
    o = V.run_world(cfg, world)
    close(y, V.expert_gemm(o["disp_x"], o["offsets"], weights, torch.bfloat16))


@pytest.mark.parametrize("E,K,T,H,N,W,zipf", [
    (8, 2, 40, 128, 128, 1, False),      # one block each way
    (64, 4, 128, 512, 384, 8, False),    # decode-like: 8 rows per expert
    (16, 4, 300, 384, 256, 4, True),     # skewed: empty experts and long segments
    (8, 2, 1200, 256, 256, 2, False),    # 300 rows per expert
    (4, 2, 1100, 1024, 384, 1, True),    # eight K blocks, three 128-column tiles, long ragged segments
    (3, 1, 700, 640, 128, 1, False),     # five K blocks: the three-buffer loop ends on its second tail step
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("fp8_rows", [False, True], ids=["rows16", "rows8"])
@pytest.mark.parametrize("padded", [False, True], ids=["compact", "padded"])
@pytest.mark.parametrize("tile", ["32", "32r", "128", "128f", "256"],
                         ids=["tile32", "tile32staged", "tile128", "tile128fourwaves", "tile256"])
def test_expert_gemm_block_quantised_weights(gpu_device, options, E, K, T, H, N, W, zipf, dtype, fp8_rows,
                                             padded, tile):
    """Weights as e4m3fn bytes with one scale per 128 x 128 block, rows 16-bit or from the fp8
    dispatch, against an f32 matmul of the dequantised operands (each rounded once to the 16-bit
    type, as two of the kernels do), through the weight-streaming kernel, the fp8 x fp8 kernel (tile
    128, fp8 rows only: 16-bit rows keep the default choice) and the 256 x 256 kernel (which needs
    N >= 256; the one N == 128 case stays on the other).  The weight-streaming form exists twice:
    slabs sent memory -> LDS directly (tile32) and staged through registers (tile32staged)."""
    options.set("GEMM_TILE", tile[:2] if tile.startswith("32") else tile[:3])
    if tile == "32r":
        options.set("GEMM_STAGED", 1)
    if tile == "128f":  # the four-wave 128 x 128 form of the fp8 x fp8 kernel (eight waves on 256 x 128 otherwise)
        options.set("GEMM_STAGED", 2)
    cfg, world, weights = make(E, K, T, H, N, W, dtype, seed=5 * E + T, zipf=zipf)
    wq, ws = V.quantize_weights_fp8(weights)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, W, fp8_dispatch=fp8_rows, padded=padded, max_recv=T if padded else None)
    d = ata.dispatch(x, idx, rs)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device))
    torch.cuda.synchronize()
    o = V.run_world(cfg, world, fp8=fp8_rows)
    # fp8 rows on segments of more than 32 rows take the fp8 x fp8 kernel unless another is forced: no
    # rounding of the rows there
    f8_kernel = fp8_rows and (tile in ("128", "128f") or (tile == "256" and N < 256 and d.num_rows > 32 * E))
    want = V.expert_gemm_q8(o["disp_x"], o["disp_scale"] if fp8_rows else None, wq, ws, o["offsets"], dtype,
                            round_rows=not f8_kernel)
    rows = d.slot_of_entry.long() if padded else o["slot_of_entry"].long().to(gpu_device)
    close(y[rows], want[o["slot_of_entry"].long()])


@pytest.mark.parametrize("E,K,T,H,N,W,zipf", [
    (8, 2, 40, 128, 128, 1, False),      # 10 rows per expert: half tiles, one 128-column block
    (4, 2, 300, 256, 256, 1, False),     # 150 rows per expert: half tiles
    (16, 4, 300, 384, 384, 4, True),     # skewed: empty experts, long segments, a 128-column tail tile
    (8, 2, 1200, 256, 512, 2, False),    # 300 rows per expert
    (3, 1, 1000, 1024, 256, 1, False),   # 333 rows per expert, eight K blocks
    (5, 2, 700, 768, 640, 1, True),      # twelve slabs of 64 bytes, a 128-column tail tile, ragged
    (2, 1, 300, 8192, 256, 1, False),    # 64 scale blocks per row: the eight-wave form's exponent table is full
    (2, 1, 300, 8448, 256, 1, False),    # 66: beyond it (the four-wave forms run)
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("padded", [False, True], ids=["compact", "padded"])
@pytest.mark.parametrize("form", [4, 3, 2, 1], ids=["eight", "eight-256-rows", "direct", "staged"])
def test_expert_gemm_power_of_two_scales(gpu_device, options, E, K, T, H, N, W, zipf, dtype, padded, form):
    """fp8 rows and fp8 weights whose scales are powers of two, multiplied by the fp8 matrix
    instruction with the scales as its block exponents, against the f32 matmul of the
    dequantised operands; the fp8 x fp8 kernel with the fold on the vector units, which takes
    any f32 scale, has to agree with it to f32 summation order.  All forms of the tiled kernel:
    eight waves on slabs of 128 columns (hidden sizes from 256; with and without the early requests for the
    rows of the weights that short segments get by themselves), four waves with slabs of 64 columns
    sent memory -> LDS directly (multiples of 256) and staged through registers (every hidden size)."""
    options.set("GEMM_TILE", "256")  # the tiles at every segment length
    options.set("GEMM_STAGED", form)
    cfg, world, weights = make(E, K, T, H, N, W, dtype, seed=7 * E + T, zipf=zipf)
    wq, ws = V.quantize_weights_fp8(weights, pow2=True)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, W, fp8_dispatch="pow2", padded=padded, max_recv=T if padded else None)
    d = ata.dispatch(x, idx, rs)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True)
    options.set("GEMM_TILE", 0)
    y_auto = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True)  # library's choice
    y_fold = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device))
    torch.cuda.synchronize()
    o = V.run_world(cfg, world, fp8=True, pow2=True)
    want = V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False)
    rows = d.slot_of_entry.long() if padded else o["slot_of_entry"].long().to(gpu_device)
    close(y[rows], want[o["slot_of_entry"].long()])
    close(y[rows], y_fold[rows].cpu())
    close(y_auto[rows], want[o["slot_of_entry"].long()])


@pytest.mark.parametrize("form", ["16bit-32", "16bit-128", "16bit-256", "q8-32", "q8-32staged", "q8-128", "q8-256",
                                  "mx-eight", "mx-early", "mx-direct", "mx-staged"])
def test_padded_overflow_stays_inside_the_buffers(gpu_device, options, form):
    """Padded layout with a LAST expert that receives more rows than max_recv (routing folds the
    surplus onto the segment's last row and raises the overflow bit; counts stay the true numbers):
    every GEMM form multiplies only the max_recv rows the segment holds.  Guard rows behind the
    output keep their sentinel, the rows of the other experts and the unfolded rows of the full
    expert equal the reference."""
    from kernel_amd import _lib

    E, K, T, H, N, W, max_recv = 8, 2, 300, 256, 256, 2, 96
    dtype = torch.bfloat16
    cfg, world, weights = make(E, K, T, H, N, W, dtype, seed=11)
    world[0].indices[:, 1] = E - 1  # every token also goes to the last expert: 300 rows for 96 places
    world[0].indices[:, 0] %= E - 1
    kind, tile = form.split("-")
    options.set("GEMM_TILE", int(tile[:3].rstrip("sd")) if tile[0].isdigit() else 256)
    if tile in ("32staged", "staged"):
        options.set("GEMM_STAGED", 1)
    if tile == "direct":
        options.set("GEMM_STAGED", 2)
    if tile in ("eight", "early"):  # the eight-wave loop without / with the early requests for the weight rows
        options.set("GEMM_STAGED", 4 if tile == "eight" else 3)
    fp8 = {"16bit": False, "q8": True, "mx": "pow2"}[kind]
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, W, fp8_dispatch=fp8, padded=True, max_recv=max_recv)
    d = ata.dispatch(x, idx, rs)
    rows = E * max_recv
    guard = 2 * max_recv + 300  # more than the surplus of the overflowing expert
    buf = torch.full((rows + guard, N), 7.0, dtype=dtype, device=gpu_device)
    if kind == "16bit":
        ata.expert_gemm(d, weights.to(gpu_device), out=buf[:rows])
    else:
        wq, ws = V.quantize_weights_fp8(weights, pow2=kind == "mx")
        ata.expert_gemm(d, wq.to(gpu_device), out=buf[:rows], w_scale=ws.to(gpu_device), scales_pow2=kind == "mx")
    torch.cuda.synchronize()
    assert int(d.status.item()) == _lib.STATUS_OVERFLOW
    assert int(d.counts[E - 1]) == T  # the true number, beyond the segment
    assert bool((buf[rows:] == 7.0).all()), "rows behind the output buffer were written"
    # reference: the same product on the rows the padded buffers hold
    dx = d.disp_x.cpu()
    sc = d.disp_scale.cpu() if fp8 else None
    counts = d.counts.cpu().clamp(max=max_recv)
    for e in range(E):
        n = int(counts[e]) - (1 if e == E - 1 else 0)  # the folded entries race for the full segment's last row
        lo = e * max_recv
        seg = torch.tensor([0, n], dtype=torch.int32)
        if kind == "16bit":
            want = V.expert_gemm(dx[lo:lo + n], seg, weights[e:e + 1], dtype)
        else:
            want = V.expert_gemm_q8(dx[lo:lo + n], sc[lo:lo + n], wq[e:e + 1], ws[e:e + 1], seg, dtype,
                                    round_rows=False)
        close(buf[lo:lo + n], want)


def test_dispatch_gemm_combine_end_to_end(gpu_device):
    """dispatch -> expert GEMM (H -> H) -> combine against the same chain on the CPU."""
    cfg, world, weights = make(32, 4, 512, 256, 256, 8, torch.bfloat16, seed=3)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 8, combine_mode=C.COMBINE_F32)
    d = ata.dispatch(x, idx, rs)
    y = ata.combine(None, w, d, ata.expert_gemm(d, weights.to(gpu_device)))
    o = V.run_world(cfg, world)
    ey = V.expert_gemm(o["disp_x"], o["offsets"], weights, torch.bfloat16)
    want = V.combine_f32(ey, w.cpu(), o["slot_of_entry"], torch.bfloat16)
    close(y, want)


@pytest.mark.parametrize("T,E", [(2048, 8), (96, 32)], ids=["wide", "skinny"])
def test_dispatch_gemm_combine_graph_replay(gpu_device, options, T, E):
    """dispatch -> expert GEMM -> combine captured once into a hipGraph; every replay, with eager
    work and synchronisation between the replays and fresh inputs each time, equals the eager
    result bit for bit (no launch of the chain allocates, clears memory or reads a value back)."""
    options.set("GEMM_TILE", 0)
    cfg, world, weights = make(E, 2, T, 256, 256, 4, torch.bfloat16, seed=T)
    x, idx, w, rs = concat_world(world, gpu_device)
    wd = weights.to(gpu_device)

    def chain(a, xx, ii, ww, out_gemm, out):
        d = a.dispatch(xx, ii, rs)
        return a.combine(out, ww, d, a.expert_gemm(d, wd, out=out_gemm))

    ata = HipAllToAll(cfg, 0, 4, combine_mode=C.COMBINE_F32)
    sx, sidx, sw = x.clone(), idx.clone(), w.clone()  # static inputs of the graph
    R = T * 2
    g_gemm = torch.empty(R, 256, dtype=torch.bfloat16, device=gpu_device)
    g_out = torch.empty(T, 256, dtype=torch.bfloat16, device=gpu_device)
    for _ in range(2):  # both buffer sets of the host class exist, first-call set-up is done
        chain(ata, sx, sidx, sw, g_gemm, g_out)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        chain(ata, sx, sidx, sw, g_gemm, g_out)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_static = chain(ata, sx, sidx, sw, g_gemm, g_out)
    eager = HipAllToAll(cfg, 0, 4, combine_mode=C.COMBINE_F32)
    gen = torch.Generator().manual_seed(3)
    for it in range(4):
        perm = torch.randperm(T, generator=gen).to(gpu_device)
        nx, nidx, nw = x[perm].contiguous(), idx[perm].contiguous(), w[perm].contiguous()
        e_gemm = torch.empty_like(g_gemm)
        want = chain(eager, nx, nidx, nw, e_gemm, None).clone()  # eager work between replays
        torch.cuda.synchronize()
        sx.copy_(nx)
        sidx.copy_(nidx)
        sw.copy_(nw)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y_static.view(torch.int16), want.view(torch.int16)), f"replay {it}"


def test_expert_gemm_argument_checks(gpu_device):
    cfg, world, weights = make(8, 2, 16, 64, 64, 1, torch.bfloat16, seed=1)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1)
    d = ata.dispatch(x, idx)
    with pytest.raises(ValueError):
        ata.expert_gemm(d, weights[:, :, :32].contiguous().to(gpu_device))
    bad = HipAllToAll(C.MoEConfig(8, 2, 72, 17, torch.bfloat16, torch.bfloat16), 0, 1)
    xb = torch.randn(16, 72, device=gpu_device).to(torch.bfloat16)
    db = bad.dispatch(xb, idx)
    from kernel_amd._lib import MoeA2AError
    with pytest.raises(MoeA2AError):  # hidden size must be a multiple of 64
        bad.expert_gemm(db, torch.zeros(8, 64, 72, dtype=torch.bfloat16, device=gpu_device))


@pytest.mark.parametrize("seed", range(20))
def test_random_shapes_every_expert_gemm_form(gpu_device, options, seed):
    """Seeded sweep: random expert counts, segment lengths (empty experts, segments that end a
    row or two past a tile), hidden and output sizes, layouts, element types, and every operand
    format (16-bit, fp8 rows, fp8 block-quantised weights, both) through whichever kernel the
    library picks for the shape and, on odd seeds, through a forced one."""
    g = torch.Generator().manual_seed(1000 + seed)

    def pick(choices):
        return choices[int(torch.randint(len(choices), (1,), generator=g))]

    E = pick([1, 3, 8, 9, 24, 40])
    K = pick([1, 2, 4])
    K = min(K, E)
    T = pick([1, 7, 33, 129, 260, 600, 1100])
    H = pick([128, 256, 384, 640])
    N = pick([128, 256, 384, 512, 640])
    W = pick([w for w in (1, 2, 4, 8) if E % w == 0])
    dtype = pick([torch.bfloat16, torch.float16])
    zipf = pick([False, True])
    padded = pick([False, True])
    fp8_rows = pick([False, True])
    q8 = pick([False, True])
    pow2 = pick([False, True]) and fp8_rows and q8  # scales as the matrix instruction's block exponents
    if seed % 2:
        options.set("GEMM_TILE", pick(["32", "128", "256"]))
    else:
        options.set("GEMM_TILE", 0)
    cfg, world, weights = make(E, K, T, H, N, W, dtype, seed=seed, zipf=zipf)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, W, fp8_dispatch="pow2" if pow2 else fp8_rows, padded=padded,
                      max_recv=T if padded else None)
    d = ata.dispatch(x, idx, rs)
    o = V.run_world(cfg, world, fp8=fp8_rows, pow2=pow2)
    if q8:
        wq, ws = V.quantize_weights_fp8(weights, pow2=pow2)
        y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=pow2)
        # which of the q8 kernels ran decides whether fp8 rows were rounded to 16 bits first; both
        # readings of the rows differ by far less than the tolerance, so the unrounded one serves
        want = V.expert_gemm_q8(o["disp_x"], o["disp_scale"] if fp8_rows else None, wq, ws, o["offsets"], dtype,
                                round_rows=False)
    elif fp8_rows:
        y = ata.expert_gemm(d, weights.to(gpu_device))
        want = V.expert_gemm_fp8(o["disp_x"], o["disp_scale"], o["offsets"], weights, dtype)
    else:
        y = ata.expert_gemm(d, weights.to(gpu_device))
        want = V.expert_gemm(o["disp_x"], o["offsets"], weights, dtype)
    torch.cuda.synchronize()
    rows = d.slot_of_entry.long() if padded else o["slot_of_entry"].long().to(gpu_device)
    close(y[rows], want[o["slot_of_entry"].long()])


def make_counts(counts, H, N, dtype, seed):
    """One rank, one expert per token, expert e receiving exactly counts[e] rows (shuffled)."""
    g = torch.Generator().manual_seed(seed)
    E = len(counts)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(ids.numel(), generator=g)].to(torch.int32).reshape(-1, 1)
    T = ids.shape[0]
    cfg = C.MoEConfig(E, 1, H, T + 1, dtype, dtype)
    world = [C.RankData(T, ids, torch.rand(T, 1, generator=g), torch.randn(T, H, generator=g).to(dtype))]
    weights = (torch.randn(E, N, H, generator=g) / H ** 0.5).to(dtype)
    return cfg, world, weights


def walk_cases():
    lone = [0, 0, 0, 3500, 0]                       # fourteen m-tiles of one expert: several groups of four
    gaps = [0] * 64
    for e, n in ((1, 256), (2, 257), (17, 1025), (18, 1), (40, 255), (63, 513)):
        gaps[e] = n                                 # tile-exact, one past a tile, one row, runs of empty experts
    many = [0] * 1024
    for e in range(0, 1024, 3):
        many[e] = 1 + (e * 7) % 5                   # the largest expert count: a few rows on every third
    many[1023] = 700
    ends = [300] + [0] * 30 + [300]                 # rows only on the first and the last expert
    return [("lone", lone), ("gaps", gaps), ("many", many), ("ends", ends)]


@pytest.mark.parametrize("name,counts", walk_cases(), ids=[c[0] for c in walk_cases()])
@pytest.mark.parametrize("fmt", ["16bit", "16bit-256-rows", "mx", "mx-256-rows", "f32scale"])
@pytest.mark.parametrize("N", [256, 640])
def test_eight_wave_tile_walk_on_odd_segment_tables(gpu_device, options, name, counts, fmt, N):
    """The eight-wave kernels give every expert's m-tiles to one die's workgroups, in groups of at
    most four.  Segment tables that stress that walk: one expert with many tiles, tile-exact and
    one-row segments between runs of empty experts, the largest expert count, rows only at the two
    ends; one n-tile and a ragged last n-tile; each operand format's eight-wave kernel forced, the two that have
    tiles of 288 rows with these wherever they save one and without."""
    dtype, H = torch.bfloat16, 256
    fmt, _, plain = fmt.partition("-")
    options.set("GEMM_TILE", "128" if fmt == "f32scale" else "256")
    if fmt != "f32scale":
        options.set("GEMM_STAGED", 3 if plain else 4)
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=len(counts) + N)
    x, idx, w, rs = concat_world(world, gpu_device)
    fp8 = {"16bit": False, "mx": "pow2", "f32scale": True}[fmt]
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch=fp8)
    d = ata.dispatch(x, idx, rs)
    o = V.run_world(cfg, world, fp8=bool(fp8), pow2=fmt == "mx")
    assert o["offsets"].tolist() == torch.tensor([0] + counts).cumsum(0).tolist()
    if fmt == "16bit":
        y = ata.expert_gemm(d, weights.to(gpu_device))
        want = V.expert_gemm(o["disp_x"], o["offsets"], weights, dtype)
    else:
        wq, ws = V.quantize_weights_fp8(weights, pow2=fmt == "mx")
        y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=fmt == "mx")
        want = V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False)
    torch.cuda.synchronize()
    close(y, want)


@pytest.mark.parametrize("H,N", [(256, 256), (384, 640), (512, 640), (640, 256), (1408, 128)])  # two, three, four, five and
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])  # eleven slabs; half a tile
def test_expert_gemm_f32_scales_wide_tiles(gpu_device, options, dtype, H, N):
    """fp8 rows and weights with f32 scales on 256 x 256 tiles: segments of 1 row, at, below and above a wave's half
    (64 rows), a wave (128), 192 and a tile (256), and several tiles.  The partial sums are folded block by block in the
    order of the 256 x 128 tiles: the same bits, and the f32 matmul within the tolerance of the other forms."""
    counts = [1, 64, 65, 0, 127, 128, 129, 192, 193, 255, 256, 257, 0, 700, 5]
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=H + N)
    wq, ws = V.quantize_weights_fp8(weights)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch=True)
    d = ata.dispatch(x, idx, rs)
    options.set("GEMM_TILE", 128)
    options.set("GEMM_STAGED", 4)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device)).clone()
    options.set("GEMM_STAGED", 5)
    y_narrow = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y_narrow.view(torch.int16))
    o = V.run_world(cfg, world, fp8=True)
    close(y, V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False))


@pytest.mark.parametrize("counts", [[1, 64, 65, 128, 129, 193, 256, 257, 0, 300], [1]], ids=["segments", "one-row"])
@pytest.mark.parametrize("H", [256, 384, 512, 640, 768, 896, 1024])  # the rows' scales come in groups of four slabs: less than
def test_expert_gemm_f32_scales_slab_groups(gpu_device, options, H, counts):  # a group, and remainders 0..3
    """fp8 with f32 scales on 256 x 256 tiles around the groups in which the rows' scales travel (rows of scales off the grid
    of 16 bytes among them), against the 256 x 128 tiles, which take them slab by slab: the same bits."""
    N, dtype = 384, torch.bfloat16
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=H)
    wq, ws = V.quantize_weights_fp8(weights)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch=True)
    d = ata.dispatch(x, idx, rs)
    options.set("GEMM_TILE", 128)
    options.set("GEMM_STAGED", 4)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device)).clone()
    options.set("GEMM_STAGED", 5)
    y_narrow = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y_narrow.view(torch.int16))
    o = V.run_world(cfg, world, fp8=True)
    close(y, V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False))


@pytest.mark.parametrize("rows", [20, 22, 23, 25, 26, 32, 33])
@pytest.mark.parametrize("form,E,H,N", [("16bit", 64, 2880, 3072), ("16bit", 64, 3072, 2944), ("16bit", 65, 512, 520),
                                        ("fp8", 65, 512, 512), ("fp8", 33, 512, 256), ("pow2", 65, 512, 512)])
def test_either_side_of_the_streaming_kernels(gpu_device, form, E, H, N, rows):
    """Mean lengths around where the library goes over from the kernels for a handful of rows to tiles of 256 rows."""
    dtype = torch.bfloat16
    counts = [rows + (e * 7) % 5 - 2 for e in range(E)]
    counts[-1] += rows * E - sum(counts)
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=H + rows)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch={"fp8": True, "pow2": "pow2"}.get(form, False))
    d = ata.dispatch(x, idx, rs)
    if form == "16bit":
        y = ata.expert_gemm(d, weights.to(gpu_device))
        rows_x, w32 = d.disp_x.float(), weights.to(gpu_device).float()
    else:
        wq, ws = V.quantize_weights_fp8(weights, pow2=form == "pow2")
        y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=form == "pow2")
        o = V.run_world(cfg, world, fp8=True, pow2=form == "pow2")
        close(y, V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False))
        return
    off = d.offsets.tolist()
    want = torch.cat([rows_x[off[e]:off[e + 1]] @ w32[e].T for e in range(E)])  # f32 on the GPU
    close(y, want.cpu())


@pytest.mark.parametrize("rows", [8, 23, 25, 32])
@pytest.mark.parametrize("E,H,N", [(65, 512, 512), (129, 256, 256), (8, 640, 128)])
def test_short_segments_take_any_scale(gpu_device, E, H, N, rows):
    """Up to 32 rows per expert the entry point for power-of-two scales multiplies with scales as they are: the bits of the one
    for any f32 scale."""
    dtype = torch.bfloat16
    cfg, world, weights = make_counts([rows] * E, H, N, dtype, seed=E + rows)
    wq, ws = V.quantize_weights_fp8(weights)  # scales with a mantissa
    assert bool((torch.frexp(ws)[0] != 0.5).any())
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch=True)
    d = ata.dispatch(x, idx, rs)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True).clone()
    y_any = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y_any.view(torch.int16))
    o = V.run_world(cfg, world, fp8=True)
    close(y, V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False))


def launched(lib, call):
    """Names of the kernels that call() launches."""
    import ctypes
    assert lib.moe_a2a_timer_begin(8) == 0
    assert call() == 0
    torch.cuda.synchronize()
    ids, us = (ctypes.c_int * 8)(), (ctypes.c_float * 8)()
    return [lib.moe_a2a_kernel_name(ids[i]).decode() for i in range(lib.moe_a2a_timer_end(ids, us, 8))]


@pytest.mark.parametrize("E,Kd,N,kernels", [
    (64, 2880, 3072, {16: "expert_gemm_skinny", 17: "expert_gemm_wide", 21: "expert_gemm_wide"}),  # 1.05 GiB of weights
    (64, 3072, 2944, {25: "expert_gemm_skinny", 26: "expert_gemm_wide"}),  # 1.08 GiB, the rows on the grid of 128 columns
    (8, 576, 512, {16: "expert_gemm_skinny", 17: "expert_gemm", 32: "expert_gemm", 33: "expert_gemm_wide"}),
    (8, 512, 512, {32: "expert_gemm_skinny", 33: "expert_gemm_wide"}),
])
def test_16bit_kernel_by_rows_per_expert(gpu_device, E, Kd, N, kernels):
    lib = _lib.load()
    w = torch.zeros(E, N, Kd, dtype=torch.bfloat16, device=gpu_device)
    for rows, name in kernels.items():
        R = rows * E
        x = torch.zeros(R, Kd, dtype=torch.bfloat16, device=gpu_device)
        y = torch.empty(R, N, dtype=torch.bfloat16, device=gpu_device)
        off = torch.arange(0, R + 1, rows, dtype=torch.int32, device=gpu_device)
        assert launched(lib, lambda: lib.moe_a2a_expert_gemm(x.data_ptr(), w.data_ptr(), off.data_ptr(), y.data_ptr(), R, E, Kd, N,
                                                             0, _lib.BF16, torch.cuda.current_stream().cuda_stream)) == [name], rows


@pytest.mark.parametrize("staged,rows,name", [(0, 22, "expert_gemm_skinny"), (0, 25, "expert_gemm_f8"), (3, 25, "expert_gemm_f8"),
                                              (4, 25, "expert_gemm_f8"), (5, 25, "expert_gemm_f8"),
                                              (1, 25, "expert_gemm_skinny"), (2, 25, "expert_gemm_skinny"),
                                              (2, 33, "expert_gemm_f8")])
@pytest.mark.parametrize("entry", ["q8", "mx8"])
def test_fp8_kernel_by_rows_per_expert_and_option(gpu_device, options, entry, staged, rows, name):
    """The options that force a form of the eight-wave tiles leave them where they are taken by default; those of the four-wave
    and register-staged forms leave the border of 32 rows."""
    lib, E, Kd, N = _lib.load(), 65, 512, 512
    if entry == "mx8" and rows > 32:
        name = "expert_gemm_mx"
    options.set("GEMM_STAGED", staged)
    R = rows * E
    x = torch.zeros(R, Kd, dtype=torch.uint8, device=gpu_device)
    w = torch.zeros(E, N, Kd, dtype=torch.uint8, device=gpu_device)
    xs, ws = torch.ones(R, Kd // 128, device=gpu_device), torch.ones(E, N // 128, Kd // 128, device=gpu_device)
    y = torch.empty(R, N, dtype=torch.bfloat16, device=gpu_device)
    off = torch.arange(0, R + 1, rows, dtype=torch.int32, device=gpu_device)
    f = getattr(lib, "moe_a2a_expert_gemm_" + entry)
    assert launched(lib, lambda: f(x.data_ptr(), xs.data_ptr(), w.data_ptr(), ws.data_ptr(), off.data_ptr(), y.data_ptr(), R, E,
                                   Kd, N, 0, _lib.BF16, torch.cuda.current_stream().cuda_stream)) == [name]


STREAM_COUNTS = {"one": [1], "runs": [33, 0, 0, 97, 32], "last": [0] * 17 + [5], "popular": [1] * 9 + [500, 0, 64, 65]}


@pytest.mark.parametrize("counts", STREAM_COUNTS.values(), ids=STREAM_COUNTS.keys())
@pytest.mark.parametrize("slabs", [1, 2, 3, 5])  # the loops take three at a time
@pytest.mark.parametrize("rows,ntile", [("16bit", 1), ("16bit", 5), ("w8", 1), ("w8", 3), ("fp8", 1), ("fp8", 3)])
def test_streaming_kernels_cover_every_tile(gpu_device, options, rows, ntile, slabs, counts):
    """The kernels for a handful of rows per expert deal their tiles out in runs: fewer tiles than runs, counts that the runs
    do not divide, several tiles of one stripe of weights, and every remainder of the loop over K."""
    dtype = torch.bfloat16
    H, N = (64 * slabs, 64 * ntile - 8) if rows == "16bit" else (128 * slabs, 128 * ntile)
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=H + N)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch=rows == "fp8")
    d = ata.dispatch(x, idx, rs)
    options.set("GEMM_TILE", 32)
    if rows == "16bit":
        y = ata.expert_gemm(d, weights.to(gpu_device))
        o = V.run_world(cfg, world)
        close(y, V.expert_gemm(o["disp_x"], o["offsets"], weights, dtype))
    else:
        wq, ws = V.quantize_weights_fp8(weights)
        y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device))
        o = V.run_world(cfg, world, fp8=rows == "fp8")
        close(y, V.expert_gemm_q8(o["disp_x"], o.get("disp_scale") if rows == "fp8" else None, wq, ws, o["offsets"], dtype,
                                  round_rows=False))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("form", ["16bit", "fp8", "pow2"])
def test_results_stored_non_temporally(gpu_device, options, form, dtype):
    """More than 256 MiB of weights under segments of less than 192 rows: the tiles of 256 rows store their results past the
    caches.  The same bits as from half of the experts at a time, whose results are stored as usual, and the f32 product."""
    H, lengths = 1024, [60, 1, 64, 65, 129, 47, 96, 31]
    E, per = (144, 2) if form == "16bit" else (272, 1)
    N = H
    assert E * N * H * per > 256 << 20
    counts = [lengths[e % 8] for e in range(E)]
    pow2 = form == "pow2"
    g = torch.Generator(device=gpu_device).manual_seed(5)
    w = torch.randn(E, N, H, device=gpu_device, generator=g)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    if form == "16bit":
        w = w.to(dtype)
        w32 = w.float()
    else:
        w = (w * 64).clamp_(-448, 448).to(torch.float8_e4m3fn)
        scale = lambda *shape: (torch.exp2(torch.randint(-7, -5, shape, device=gpu_device, generator=g).float()) if pow2
                                else 0.01 * (1 + torch.rand(shape, device=gpu_device, generator=g)))
        ws = scale(E, N // 128, H // 128)
        w32 = w.float() * ws.repeat_interleave(128, 1).repeat_interleave(128, 2)
    R = sum(counts)
    x = torch.randn(R, H, device=gpu_device, generator=g)
    if form == "16bit":
        x = x.to(dtype)
        x32 = x.float()
    else:
        x = (x * 64).clamp_(-448, 448).to(torch.float8_e4m3fn)
        xs = scale(R, H // 128)
        x32 = x.float() * xs.repeat_interleave(128, 1)
    options.set("GEMM_TILE", 256 if form != "fp8" else 128)
    options.set("GEMM_STAGED", 3)

    def product(rows, off, experts, first):
        y = torch.empty(rows, N, dtype=dtype, device=gpu_device)
        et = _lib.BF16 if dtype == torch.bfloat16 else _lib.F16
        tail = (off.data_ptr(), y.data_ptr(), rows, experts, H, N, 0, et, stream)
        if form == "16bit":
            rc = lib.moe_a2a_expert_gemm(x.data_ptr(), w[first].data_ptr(), *tail)
        else:
            f = lib.moe_a2a_expert_gemm_mx8 if pow2 else lib.moe_a2a_expert_gemm_q8
            rc = f(x.data_ptr(), xs.data_ptr(), w[first].data_ptr(), ws[first].data_ptr(), *tail)
        assert rc == 0
        return y

    off = torch.tensor([0] + counts, device=gpu_device).cumsum(0).to(torch.int32)
    y = product(R, off, E, 0)
    # half of the experts at a time: less than 256 MiB, stored as usual (the offsets of the second half start behind the first)
    h, mid = E // 2, int(off[E // 2])
    usual = torch.cat([product(R, off[:h + 1].contiguous(), h, 0)[:mid], product(R, off[h:].contiguous(), E - h, h)[mid:]])
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), usual.view(torch.int16))
    o = off.tolist()
    want = torch.cat([x32[o[e]:o[e + 1]] @ w32[e].T for e in range(E)])
    close(y, want.cpu())


TALL_COUNTS = [1, 255, 256, 257, 0, 272, 273, 287, 288, 289, 512, 513, 544, 545, 576, 577, 864, 865]


@pytest.mark.parametrize("H,N", [(192, 256), (256, 640), (320, 200)])  # N: one tile, a ragged last one, less than one
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_expert_gemm_16bit_tall_tiles(gpu_device, options, dtype, H, N):
    """Segments at and around the lengths where tiles of 288 rows save one of 256: every 16-bit kernel walks K in the
    same order, so the 128 x 128 tiles give the same bits."""
    cfg, world, weights = make_counts(TALL_COUNTS, H, N, dtype, seed=H + N)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1)
    d = ata.dispatch(x, idx, rs)
    options.set("GEMM_TILE", 256)
    options.set("GEMM_STAGED", 4)
    y = ata.expert_gemm(d, weights.to(gpu_device)).clone()
    options.set("GEMM_TILE", 128)
    y_small = ata.expert_gemm(d, weights.to(gpu_device))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y_small.view(torch.int16))
    o = V.run_world(cfg, world)
    close(y, V.expert_gemm(o["disp_x"], o["offsets"], weights, dtype))


@pytest.mark.parametrize("H,N", [(256, 256), (384, 640), (1408, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_expert_gemm_power_of_two_tall_tiles(gpu_device, options, dtype, H, N):
    """The same segments through the kernel with power-of-two scales, with the same bits as with tiles of 256 rows only."""
    cfg, world, weights = make_counts(TALL_COUNTS, H, N, dtype, seed=H + N)
    wq, ws = V.quantize_weights_fp8(weights, pow2=True)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch="pow2")
    d = ata.dispatch(x, idx, rs)
    options.set("GEMM_TILE", 256)
    options.set("GEMM_STAGED", 4)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True).clone()
    options.set("GEMM_STAGED", 3)
    y_short = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y_short.view(torch.int16))
    o = V.run_world(cfg, world, fp8=True, pow2=True)
    close(y, V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False))


@pytest.mark.parametrize("H", [4224, 4608, 8192])  # 33 (four by four does not go), 36 and 64 slabs
def test_expert_gemm_power_of_two_exponent_table(gpu_device, options, H):
    """Rows of more scales than are requested ahead of the operands, and of the most that the table holds, with and without
    the rows behind a tile's 256th: the same bits from both tilings, and the oracle's results."""
    counts, N, dtype = [1, 65, 0, 129, 256, 257, 288, 300], 256, torch.bfloat16
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=H)
    wq, ws = V.quantize_weights_fp8(weights, pow2=True)
    x, idx, w, rs = concat_world(world, gpu_device)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch="pow2")
    d = ata.dispatch(x, idx, rs)
    options.set("GEMM_TILE", 256)
    options.set("GEMM_STAGED", 4)
    y = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True).clone()
    options.set("GEMM_STAGED", 3)
    y_plain = ata.expert_gemm(d, wq.to(gpu_device), w_scale=ws.to(gpu_device), scales_pow2=True)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y_plain.view(torch.int16))
    o = V.run_world(cfg, world, fp8=True, pow2=True)
    close(y, V.expert_gemm_q8(o["disp_x"], o["disp_scale"], wq, ws, o["offsets"], dtype, round_rows=False))


def tall_tiles_pay(counts, ntile_n):
    """The kernels' rule: whether tall tiles save some, and whether the plan with them is the faster one by their estimate."""
    R, plain, tall = sum(counts), sum(-(-c // 256) for c in counts), sum(-(-c // 288) for c in counts)
    rounds = {n: -(-(-(-n // 8) * ntile_n) // 32) for n in (plain, tall)}
    if max(counts) * len(counts) > 2.5 * R:
        pays = 1.1 * rounds[tall] < rounds[plain]
    else:
        pays = (288 * tall + R) * rounds[tall] / tall < (288 * plain + R) * rounds[plain] / plain
    return tall < plain, pays


SKEWED = {  # segment tables where tall tiles save some, and whether the kernels take them (8 n-tiles)
    "popular-tall": ([min(1500, int(1500 / (e + 1) ** 1.2)) for e in range(24)], True),
    "popular-256": ([int(2500 / (e + 1) ** 1.2) for e in range(24)], False),
    "alike-tall": ([281] * 36, True),
    "alike-256": ([257 + (e * 31) % 40 for e in range(30)], False),
    "lone-tall": ([0, 0, 8193, 0], True),
    "lone-256": ([0, 288, 0], False),
    "ends-256": ([288] + [1] * 7 + [0] * 600 + [288], False),
}


@pytest.mark.parametrize("table", SKEWED)
@pytest.mark.parametrize("fmt", ["16bit", "mx"])
def test_tall_tiles_on_skewed_segment_tables(gpu_device, options, table, fmt):
    """Tables on either side of the rule that weighs tall tiles against 256-row ones, as the kernels decide and with tall
    tiles wherever they save one: the bits of a form that has no tall tiles, and the f32 matmul within the tolerance of
    the other forms."""
    counts, tall = SKEWED[table]
    dtype, H, N = torch.bfloat16, 256, 1920
    assert tall_tiles_pay(counts, 8) == (True, tall)
    R, E = sum(counts), len(counts)
    g = torch.Generator(device=gpu_device).manual_seed(R)
    w = (torch.randn(E, N, H, device=gpu_device, generator=g) / H ** 0.5).to(dtype)
    x = torch.randn(R, H, device=gpu_device, generator=g).to(dtype)
    offsets = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    at = offsets.to(gpu_device)
    tail = (R, E, H, N, 0, _lib.BF16, torch.cuda.current_stream().cuda_stream)
    lib = _lib.load()
    if fmt == "mx":
        q, s = torch.empty(R, H, dtype=torch.uint8, device=gpu_device), torch.empty(R, H // 128, device=gpu_device)
        same = torch.arange(R, dtype=torch.int32, device=gpu_device)
        _lib.check(lib.moe_a2a_dispatch_fp8(x.data_ptr(), _lib.BF16, same.data_ptr(), q.data_ptr(), s.data_ptr(), R, 1, H,
                                            _lib.FP8_SCALE_POW2, tail[-1]), "moe_a2a_dispatch_fp8")
        wq, ws = (t.to(gpu_device) for t in V.quantize_weights_fp8(w.cpu(), pow2=True))
        x = (q.view(torch.float8_e4m3fn).float().view(R, -1, 128) * s[..., None]).view(R, H)
        w = (wq.view(torch.float8_e4m3fn).float().view(E, N // 128, 128, H // 128, 128) * ws[:, :, None, :, None]).view(E, N, H)

    def gemm(form):
        options.set("GEMM_TILE", 256)
        options.set("GEMM_STAGED", form)
        y = torch.empty(R, N, dtype=dtype, device=gpu_device)
        if fmt == "mx":
            _lib.check(lib.moe_a2a_expert_gemm_mx8(q.data_ptr(), s.data_ptr(), wq.data_ptr(), ws.data_ptr(), at.data_ptr(),
                                                   y.data_ptr(), *tail), "moe_a2a_expert_gemm_mx8")
        else:
            _lib.check(lib.moe_a2a_expert_gemm(x.data_ptr(), w.data_ptr(), at.data_ptr(), y.data_ptr(), *tail),
                       "moe_a2a_expert_gemm")
        return y

    want = torch.empty(R, N, device=gpu_device)
    for e in range(E):
        rows = slice(int(offsets[e]), int(offsets[e + 1]))
        want[rows] = x[rows].float() @ w[e].float().T
    decided, forced, none = gemm(0), gemm(4), gemm(3)
    torch.cuda.synchronize()
    assert torch.equal(decided.view(torch.int16), none.view(torch.int16))
    assert torch.equal(forced.view(torch.int16), none.view(torch.int16))
    close(forced, want.cpu())


@pytest.mark.parametrize("Kd", [3728256, 3728320, 4194240])  # the longest rows of a tall tile, one slab more, and more
def test_expert_gemm_16bit_longest_rows(gpu_device, options, Kd):
    """A segment of 288 rows, which are one tall tile, so long that the tile's offsets come to the end of 32 bits: the sum
    of every row, the last 32 among them, whatever tile they fall to.  Tolerance: one rounding to bf16 (2^-9 of a value)
    and the f32 sum of Kd products of variance 1 / Kd in any order, whose error stays below sqrt(Kd) * 2^-24 * 4 = 5e-4."""
    counts = [288] + [1] * 7
    R, E, N = sum(counts), len(counts), 8
    gen = torch.Generator(device=gpu_device).manual_seed(Kd)
    x = torch.empty(R, Kd, dtype=torch.bfloat16, device=gpu_device).normal_(generator=gen)
    w = torch.empty(E, N, Kd, dtype=torch.bfloat16, device=gpu_device).normal_(0.0, Kd ** -0.5, generator=gen)
    offsets = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32)
    y = torch.empty(R, N, dtype=torch.bfloat16, device=gpu_device)
    options.set("GEMM_TILE", 256)
    options.set("GEMM_STAGED", 4)
    at = offsets.to(gpu_device)
    _lib.check(_lib.load().moe_a2a_expert_gemm(x.data_ptr(), w.data_ptr(), at.data_ptr(), y.data_ptr(), R, E, Kd, N, 0,
                                               _lib.BF16, torch.cuda.current_stream().cuda_stream), "moe_a2a_expert_gemm")
    want = torch.zeros(R, N, dtype=torch.float64, device=gpu_device)
    for k in range(0, Kd, 1 << 16):
        for e in range(E):
            rows = slice(int(offsets[e]), int(offsets[e + 1]))
            want[rows] += (x[rows, k:k + (1 << 16)].float() @ w[e, :, k:k + (1 << 16)].float().T).double()
    assert bool(((y.double() - want).abs() <= want.abs() * 2 ** -8 + 5e-4).all())


STRIP_NAMES = {"16bit": "expert_gemm_strip", "fp8": "expert_gemm_strip_f8", "pow2": "expert_gemm_strip_mx", "w8": "expert_gemm_strip_w8"}
# rows of a segment around the forms of a strip (64, 96, 112, 128, 144, 160, 176) and of two and more of them
STRIP_COUNTS = [1, 16, 17, 64, 65, 96, 97, 112, 113, 0, 128, 129, 144, 145, 160, 161, 175, 176, 177, 352, 353, 900]


@pytest.mark.parametrize("counts", [STRIP_COUNTS, [1], [0, 0, 5]], ids=["segments", "one-row", "first-empty"])
@pytest.mark.parametrize("form,slabs,N", [("16bit", 1, 8), ("16bit", 2, 520), ("16bit", 5, 1032), ("fp8", 8, 128), ("fp8", 11, 640),
                                          ("fp8", 16, 1152), ("pow2", 9, 512), ("pow2", 15, 640), ("w8", 1, 128), ("w8", 2, 640),
                                          ("w8", 9, 1152)])
@pytest.mark.parametrize("padded", [False, True], ids=["compact", "padded"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_strips(gpu_device, options, dtype, padded, form, slabs, N, counts):
    """Tiles of 512 columns: every form of a tile, a last one of any width, one slab to several groups of scales with a rest, the
    padded layout with a segment longer than its room.  The bits of the 256 x 256 tiles, where there are such, and the f32 product."""
    H = slabs * (64 if form == "16bit" else 128)
    cfg, world, weights = make_counts(counts, H, N, dtype, seed=H + N + len(counts))
    x, idx, w, rs = concat_world(world, gpu_device)
    room = max(counts) - 1 if padded and max(counts) > 1 else max(counts)
    ata = HipAllToAll(cfg, 0, 1, fp8_dispatch={"fp8": True, "pow2": "pow2"}.get(form, False), padded=padded,
                      max_recv=room if padded else None)
    d = ata.dispatch(x, idx, rs)
    off = torch.tensor([0] + counts).cumsum(0)
    lens = [min(c, room) if padded else c for c in counts]
    rows = torch.cat([torch.arange(n) + (e * room if padded else int(off[e])) for e, n in enumerate(lens)]).to(gpu_device)
    if form == "16bit":
        wd, kw = weights.to(gpu_device), {}
        x32, w32 = d.disp_x.float(), wd.float()
    else:
        wq, ws = V.quantize_weights_fp8(weights, pow2=form == "pow2")
        wd = wq.to(gpu_device)
        kw = dict(w_scale=ws.to(gpu_device), scales_pow2=form == "pow2")
        x32 = d.disp_x.float() if form == "w8" else d.disp_x.view(torch.float8_e4m3fn).float() * d.disp_scale.repeat_interleave(128, 1)
        w32 = wd.view(torch.float8_e4m3fn).float() * kw["w_scale"].repeat_interleave(128, 1).repeat_interleave(128, 2)
    # (power-of-two scales of up to 32 rows on average take the kernels for any scale)
    strip = STRIP_NAMES["fp8" if form == "pow2" and sum(counts) <= 32 * len(counts) else form]
    got = {}
    for tile, staged in ((512, 0), (128 if form == "fp8" else 32 if form == "w8" else 256, 3)):
        options.set("GEMM_TILE", tile)
        options.set("GEMM_STAGED", staged)
        result = []
        names = launched(ata.lib, lambda: result.append(ata.expert_gemm(d, wd, **kw)) or 0)
        assert len(names) == 1 and (names[0] == strip if tile == 512 else "strip" not in names[0]), names
        got[tile] = result[0][rows].clone()
    torch.cuda.synchronize()
    want = torch.cat([x32[(first := e * room if padded else int(off[e])):first + n] @ w32[e].T for e, n in enumerate(lens)])
    close(got[512], want.cpu())
    first, second = got.values()
    # (fp8 weights: the streaming kernel walks K in another order)
    if form not in ("pow2", "w8") or (form == "pow2" and sum(counts) > 32 * len(counts)):
        assert torch.equal(first.view(torch.int16), second.view(torch.int16))


def product_of(lib, form, x, xs, w, ws, off, y):
    """y = x w^T through the form's entry point; the kernels that were launched."""
    E, N, Kd = w.shape
    tail = (off.data_ptr(), y.data_ptr(), x.shape[0], E, Kd, N, 0, _lib.BF16, torch.cuda.current_stream().cuda_stream)
    if form == "16bit":
        return launched(lib, lambda: lib.moe_a2a_expert_gemm(x.data_ptr(), w.data_ptr(), *tail))
    f = lib.moe_a2a_expert_gemm_mx8 if form == "pow2" else lib.moe_a2a_expert_gemm_q8
    return launched(lib, lambda: f(x.data_ptr(), None if form == "w8" else xs.data_ptr(), w.data_ptr(), ws.data_ptr(), *tail))


@pytest.mark.parametrize("form,rows,Kd,fits", [("16bit", 176, 2097088, True), ("16bit", 176, 2097152, False), ("fp8", 176, 4194176, True),
                                               ("pow2", 176, 4194176, True), ("w8", 160, 2097024, True)])
def test_longest_rows_of_a_strip(gpu_device, options, form, rows, Kd, fits):
    """A full strip of rows so long that its 512 rows of weights come to the end of 31 bits, and a slab more, which is left to the
    256 x 256 tiles.  x is zero but for the first and the last 128 columns, so that a row, a column or a slab that is fetched from a place
    other than its own shows.  Tolerance: one rounding to bf16, and f32 sums of 256 products, 2^-24 of their absolute sum each."""
    N = 512
    g = torch.Generator(device=gpu_device).manual_seed(Kd)
    cols = torch.cat([torch.arange(128), torch.arange(Kd - 128, Kd)]).to(gpu_device)
    part = torch.randn(rows, 256, device=gpu_device, generator=g)
    if form == "16bit":
        w = torch.empty(1, N, Kd, dtype=torch.bfloat16, device=gpu_device).normal_(generator=g)
        w32 = w[0][:, cols].float()
    else:
        w = torch.empty(1, N, Kd, dtype=torch.uint8, device=gpu_device).random_(0x20, 0x48, generator=g)  # 2^-4 .. 4, no NaN
        w32 = w[0][:, cols].view(torch.float8_e4m3fn).float()
    scales = lambda *shape: torch.exp2(torch.randint(-2, 3, shape, device=gpu_device, generator=g).float()) * (1.0 if form == "pow2" else 1.3)
    xs, ws = (scales(rows, Kd // 128), scales(1, N // 128, Kd // 128)) if form != "16bit" else (None, None)
    dtype = torch.bfloat16 if form in ("16bit", "w8") else torch.float8_e4m3fn
    part = part.to(dtype)
    x = torch.zeros(rows, Kd, dtype=torch.uint8 if dtype == torch.float8_e4m3fn else dtype, device=gpu_device)
    x[:, cols] = part.view(x.dtype)
    x32 = part.float()
    if form != "16bit":
        if form != "w8":
            x32 = x32 * xs[:, cols // 128]
        w32 = w32 * ws[0][:, cols // 128].repeat_interleave(128, 0)
    y = torch.full((rows, N), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    off = torch.tensor([0, rows], dtype=torch.int32, device=gpu_device)
    options.set("GEMM_TILE", 512)
    names = product_of(_lib.load(), form, x, xs, w, ws, off, y)
    assert names == [STRIP_NAMES[form] if fits else "expert_gemm"]
    want, size = x32.double() @ w32.double().T, x32.double().abs() @ w32.double().abs().T
    assert bool(((y.double() - want).abs() <= want.abs() * 2 ** -8 + size * 2.0 ** -16).all())


@pytest.mark.parametrize("form,E,Kd,N,kernels", [
    ("16bit", 256, 512, 1024, {15: "expert_gemm_skinny", 16: "strip", 140: "strip", 141: "expert_gemm_wide", 289: "expert_gemm_wide",
                               290: "strip", 310: "strip", 311: "expert_gemm_wide"}),
    ("16bit", 256, 512, 2048, {140: "strip", 141: "expert_gemm_wide"}),
    ("16bit", 256, 2048, 1024, {104: "strip", 105: "expert_gemm_wide"}),  # 104 MiB of rows
    ("16bit", 64, 8192, 5120, {128: "strip", 129: "expert_gemm_wide"}),  # more, 40 columns per row
    ("16bit", 256, 512, 768, {23: "expert_gemm_skinny", 24: "strip", 112: "strip", 113: "expert_gemm_wide", 300: "expert_gemm_wide"}),
    ("16bit", 255, 512, 768, {100: "expert_gemm_wide"}),
    ("fp8", 256, 1024, 1024, {15: "expert_gemm_skinny", 16: "strip", 144: "strip", 145: "expert_gemm_f8", 249: "expert_gemm_f8",
                              250: "strip", 310: "strip", 311: "expert_gemm_f8"}),
    ("fp8", 256, 1024, 768, {23: "expert_gemm_f8", 24: "strip", 120: "strip", 121: "expert_gemm_f8", 300: "expert_gemm_f8"}),
    ("fp8", 256, 1024, 512, {95: "expert_gemm_f8", 96: "strip", 128: "strip", 129: "expert_gemm_f8", 300: "expert_gemm_f8"}),
    ("fp8", 256, 896, 1536, {100: "expert_gemm_f8"}),  # less than eight slabs
    ("fp8", 255, 1024, 512, {100: "expert_gemm_f8"}),  # less than one round
    ("pow2", 256, 1024, 512, {95: "expert_gemm_mx", 96: "strip", 128: "strip", 129: "expert_gemm_mx"}),
    ("pow2", 256, 1024, 1024, {33: "strip", 140: "strip", 141: "expert_gemm_mx", 300: "expert_gemm_mx"}),
    ("pow2", 256, 1024, 4096, {144: "strip", 145: "expert_gemm_mx", 289: "expert_gemm_mx", 290: "strip", 310: "strip", 311: "expert_gemm_mx"}),
    ("w8", 256, 256, 4096, {24: "expert_gemm_skinny", 25: "strip"}),
    ("w8", 256, 256, 1024, {32: "expert_gemm_skinny", 33: "strip", 700: "strip"}),
    ("w8", 256, 256, 512, {32: "expert_gemm_skinny", 33: "strip"}),
    ("w8", 255, 256, 512, {33: "expert_gemm_wide"}),
])
def test_where_strips_are_taken(gpu_device, options, form, E, Kd, N, kernels):
    """Lengths on both sides of every border.  Products of ones."""
    lib = _lib.load()
    for rows, name in kernels.items():
        R = rows * E
        one = 0x38  # 1.0 in e4m3fn
        ones = lambda *shape: torch.ones(shape, dtype=torch.bfloat16, device=gpu_device)
        bytes_ = lambda *shape: torch.full(shape, one, dtype=torch.uint8, device=gpu_device)
        x = (ones if form in ("16bit", "w8") else bytes_)(R, Kd)
        w = (ones if form == "16bit" else bytes_)(E, N, Kd)
        xs, ws = torch.ones(R, Kd // 128, device=gpu_device), torch.ones(E, N // 128, Kd // 128, device=gpu_device)
        y = torch.zeros(R, N, dtype=torch.bfloat16, device=gpu_device)
        off = torch.arange(0, R + 1, rows, dtype=torch.int32, device=gpu_device)
        got = product_of(lib, form, x, xs, w, ws, off, y)
        assert got == [STRIP_NAMES[form] if name == "strip" else name], rows
        assert bool((y == Kd).all()), rows
