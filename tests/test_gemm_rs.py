"""GEMM + reduce-scatter (the reference's gemm_rs problem) on one GPU.

CPU: the oracle against the vectors the reference itself wrote over gloo, the C ABI of
include/gemm_rs.h (symbols, host-side argument checks), the input generator.
GPU (``-m gpu``): the HIP path through the C ABI against the reference's vectors, the oracle, the
exact f64 sum on sampled rows and an f32 matrix product of the whole output, for the reference's
test and benchmark shapes at full size and for each of the three kernel forms.

Tolerances.  The reference accepts rtol = atol = 1e-2 (gemm_rs/reference.py:66).  The HIP path
accumulates in f32 over the whole of K and rounds once, so it is also held to the exact sum within
one bf16 rounding: |out - exact| <= 2^-8 |exact| + 1e-6 (2^-9 is half a unit in the last place; the
f32 accumulation adds less than 2^-15 relative over these K).
"""
import ctypes
import random
import glob
import os
import re

import numpy as np
import pytest
import torch

from kernel_amd import _lib
from kernel_amd import gemm_rs as G
from oracle import gemm_rs as O

import tile_loops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gemm_rs.h")
GOLDEN = sorted(glob.glob(os.path.join(ROOT, "tests", "golden", "gemm_rs_*.npz")))
E_NULL, E_SHAPE, E_DTYPE, E_WORKSPACE, E_ALIGN = -1, -2, -3, -4, -5
A = 0x1000  # any non-NULL, 16-byte aligned address; never dereferenced on the host


def load_golden(path):
    d = np.load(path)
    W = int(d["world_size"])
    bf = lambda a: torch.from_numpy(a.copy()).view(torch.bfloat16)
    bias = bf(d["r0_bias"]) if int(d["has_bias"]) else None
    datas = [(bf(d[f"r{r}_input"]), bf(d[f"r{r}_weight"]), bias) for r in range(W)]
    want = torch.cat([bf(d[f"r{r}_out"]) for r in range(W)], 0)
    return datas, want


def within_one_rounding(out, exact):
    err = (out.double() - exact).abs()
    return bool((err <= exact.abs() * 2.0 ** -8 + 1e-6).all()), float(err.max())


# ---------------------------------------------------------------------------------------------
# CPU
# ---------------------------------------------------------------------------------------------
def test_golden_files_exist():
    assert len(GOLDEN) == 4


@pytest.mark.parametrize("path", GOLDEN, ids=lambda p: os.path.basename(p)[:-4])
def test_oracle_against_the_reference_vectors(path):
    datas, want = load_golden(path)
    got = O.ref_world(datas)
    assert got.shape == want.shape and got.dtype == want.dtype
    W = len(datas)
    if W == 2:  # one addition in the reduction: no order to choose, so the bits are defined
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # a quarter of the reference's own tolerance (a few bf16 units in the last place of the sum)
    assert torch.allclose(got.float(), want.float(), rtol=2.5e-3, atol=2.5e-3)
    ok, _ = O.check_implementation(want, got)
    assert ok
    # both are the exact sum up to the rounding of W bf16 products and W - 1 bf16 additions
    exact = O.exact_world(datas)
    bound = 2.0 ** -8 * (2 * W) * exact.abs().max().item() + 1e-6
    assert (want.double() - exact).abs().max().item() <= bound
    assert (got.double() - exact).abs().max().item() <= bound


def test_the_bias_enters_once_per_rank():
    """What the vectors pin and a reading could get wrong: W times the bias, not once."""
    datas, want = load_golden([p for p in GOLDEN if p.endswith("gemm_rs_w8_bias.npz")][0])
    W, bias = len(datas), datas[0][2]
    no_bias = O.exact_world([(x, w, None) for x, w, _ in datas])
    resid = (want.double() - no_bias).mean(0)  # per column: what the bias contributed
    assert torch.allclose(resid, W * bias.double(), atol=2e-4)
    assert not torch.allclose(resid, bias.double(), atol=2e-3)


def test_row_block_r_is_rank_r(tmp_path):
    datas, want = load_golden([p for p in GOLDEN if p.endswith("gemm_rs_w4_nobias.npz")][0])
    W, M = len(datas), want.shape[0]
    exact = O.exact_world(datas)
    d = np.load([p for p in GOLDEN if p.endswith("gemm_rs_w4_nobias.npz")][0])
    for r in range(W):
        mine = torch.from_numpy(d[f"r{r}_out"].copy()).view(torch.bfloat16)
        blk = exact[r * M // W:(r + 1) * M // W]
        assert mine.shape == blk.shape
        assert (mine.double() - blk).abs().max().item() <= 2.0 ** -8 * 2 * W * exact.abs().max().item() + 1e-6


def test_generate_input_follows_the_reference_distribution():
    x, w, b = G.generate_input(3, 8, 64, 96, 2880, True, 7)
    assert x.shape == (64, 360) and w.shape == (96, 360) and b.shape == (96,)
    assert x.dtype == w.dtype == b.dtype == torch.bfloat16
    assert x.abs().max().item() <= 0.0101 and w.abs().max().item() <= 0.0101  # bf16 rounds 0.00999.. up
    assert abs(x.float().mean().item()) < 2e-4 and abs(x.float().std().item() - 0.01 / 3 ** 0.5) < 3e-4
    x2, _, b2 = G.generate_input(4, 8, 64, 96, 2880, True, 7)
    assert not torch.equal(x, x2) and torch.equal(b, b2)  # the same bias on every rank
    assert G.generate_input(0, 8, 64, 96, 2880, False, 7)[2] is None
    assert len(G.TEST_SPECS) == 11 and len(G.BENCHMARK_SPECS) == 6


def declared_functions():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    return sorted(set(re.findall(r"\b(gemm_rs_[a-z0-9_]+)\s*\(", text)))


def test_header_binding_and_exports_agree():
    assert declared_functions() == sorted(_lib.GEMM_RS_PROTOTYPES)
    raw = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared_functions():
        assert hasattr(raw, name), f"{name} is declared in include/gemm_rs.h but not exported"


def test_host_side_argument_checks():
    lib = _lib.load()
    f = lib.gemm_rs_forward
    ok = dict(M=256, N=256, K=1024, W=8)
    call = lambda inp=A, wt=A, out=A, M=256, N=256, K=1024, W=8, et=_lib.BF16, ws=None, wsb=0: f(
        inp, wt, None, out, M, N, K, W, 0, 0, et, ws, wsb, None)
    assert call(K=1000) == E_SHAPE            # K not divisible by W
    assert call(K=8 * 12) == E_SHAPE          # local K not a multiple of 8
    assert call(W=0) == E_SHAPE and call(N=0) == E_SHAPE and call(M=-1) == E_SHAPE
    assert call(et=7) == E_DTYPE
    assert call(M=0) == 0                     # nothing to do, nothing launched
    assert call(inp=None) == E_NULL and call(wt=None) == E_NULL and call(out=None) == E_NULL
    assert call(inp=A + 4) == E_ALIGN
    assert f(A, A, None, A, 256, 256, 1024, 8, 100, 0, _lib.BF16, None, 0, None) == E_SHAPE  # shards would overlap
    # an output of few tiles keeps one partial product per shard and needs the workspace for them
    need = lib.gemm_rs_workspace_bytes(64, 7168, 18432, 8)
    assert need == 8 * 64 * 7168 * 4
    assert call(M=64, N=7168, K=18432) == E_WORKSPACE
    assert call(M=64, N=7168, K=18432, ws=A, wsb=need - 1) == E_WORKSPACE
    assert lib.gemm_rs_workspace_bytes(8192, 4096, 14336, 8) == 0  # whole slabs per shard, enough tiles
    # ragged shards on 256 x 256 tiles: room for both operands in rows padded to whole 64-column slabs
    # (optional: without it the product runs on the rows as they lie)
    assert lib.gemm_rs_workspace_bytes(8192, 8192, 29568, 8) == 8 * (8192 + 8192) * 3712 * 2
    # a few hundred rows: 256 x 128 tiles with the shards in four groups
    assert lib.gemm_rs_workspace_bytes(512, 4096, 12288, 8) == 4 * 512 * 4096 * 4
    assert lib.gemm_rs_workspace_bytes(64, 64, 100, 8) == 0  # invalid shape: no size


def test_bytes_told_of_and_not_used():
    """Shards off the line grid on 256 x 256 tiles: the room that gemm_rs_workspace_bytes tells of has not been used since operands were
    copied there."""
    assert _lib.load().gemm_rs_workspace_used(8192, 8192, 29568, 8) == 0


@pytest.mark.parametrize("m,n,k,groups", [
    (496, 8192, 12288, 2), (1024, 3456, 9728, 2), (720, 4736, 9216, 2),  # not one group of tiles with 128 rows in use
    (584, 2432, 24576, 4), (512, 4096, 12288, 4), (128, 4096, 16896, 8), (2048, 2880, 2880, 1), (1088, 5184, 3584, 1),
])
def test_groups_of_shards(m, n, k, groups):
    """Groups that the 256 x 128 tiles spread the shards over, by the room for their partial products: the fastest of 1, 2, 4
    and 8 where these were timed one against the other."""
    assert _lib.load().gemm_rs_workspace_bytes(m, n, k, 8) == (groups * m * n * 4 if groups > 1 else 0)


def test_no_cpu_path():
    x, w, b = G.generate_input(0, 1, 8, 8, 64, True, 1)
    with pytest.raises(RuntimeError):
        G.custom_kernel((x, w, b))


# ---------------------------------------------------------------------------------------------
# GPU
# ---------------------------------------------------------------------------------------------
def to_dev(datas, dev):
    return [(x.to(dev), w.to(dev), b.to(dev) if b is not None else None) for x, w, b in datas]


@pytest.mark.gpu
@pytest.mark.parametrize("path", GOLDEN, ids=lambda p: os.path.basename(p)[:-4])
def test_hip_against_the_reference_vectors(gpu_device, path):
    datas, want = load_golden(path)
    outs = G.custom_kernel_world(to_dev(datas, gpu_device))
    W, M = len(datas), want.shape[0]
    assert len(outs) == W and all(o.shape == (M // W, want.shape[1]) for o in outs)
    got = torch.cat(outs, 0).cpu()
    ok, msg = O.check_implementation(want, got)  # the reference's own acceptance test, on its own result
    assert ok, msg
    ok, worst = within_one_rounding(got, O.exact_world(datas))
    assert ok, worst


def spec_id(s):
    return f"m{s['m']}-n{s['n']}-k{s['k']}-{'bias' if s['has_bias'] else 'nobias'}"


@pytest.mark.gpu
@pytest.mark.parametrize("spec", G.TEST_SPECS + G.BENCHMARK_SPECS, ids=spec_id)
def test_reference_shapes_at_full_size(gpu_device, spec):
    W, m, n, k = spec["world_size"], spec["m"], spec["n"], spec["k"]
    datas = [G.generate_input(r, device=None, **spec) for r in range(W)]
    x, w, bias = G.pack_world(datas, gpu_device)
    out = G.HipGemmReduceScatter(W).forward(x, w, bias)
    torch.cuda.synchronize()
    assert out.shape == (m, n) and out.dtype == torch.bfloat16
    # (1) every element against an f32 matrix product of the concatenated shards (torch's own GEMM)
    xc = x.permute(1, 0, 2).reshape(m, k).float()
    wc = w.permute(1, 0, 2).reshape(n, k).float()
    ref = xc @ wc.T
    if bias is not None:
        ref += W * bias.float()
    assert torch.allclose(out.float(), ref, rtol=1e-2, atol=1e-2)
    err = (out.float() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 2e-6).all()), float(err.max())
    del xc, wc, ref, err
    # (2) sampled rows against the exact f64 sum on the CPU
    g = torch.Generator().manual_seed(spec["seed"])
    rows = torch.randperm(m, generator=g)[:16]
    sample = [(d[0][rows], d[1], d[2]) for d in datas]
    ok, worst = within_one_rounding(out[rows.to(gpu_device)].cpu(), O.exact_world(sample))
    assert ok, worst
    # (3) the whole oracle where it finishes in seconds
    if m * n * k <= 3e10:
        want = O.ref_world(datas)
        ok, msg = O.check_implementation(want, out.cpu())
        assert ok, msg


@pytest.mark.gpu
@pytest.mark.parametrize("form", [256, 129, 131, 132, 130, 128, 32])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("k", [1024, 1440, 4 * 72], ids=["k256", "k360", "k72"])
def test_each_kernel_form(gpu_device, options, form, dtype, k):
    """256 x 256 tiles, 256 x 128 tiles (129; 131 / 132: 192 / 128 of their rows in use, the former on
    the map that deals the tiles out evenly; 130: with per-shard partial products), 128 x 128 tiles and
    their per-shard partial products (32) on one shape with ragged
    edges (M and N not multiples of the tiles); local K a multiple of the 64-column slab, five slabs
    and a short one (360: the wide tiles start the last slab of a shard early and mask what it
    shares with the one before), and one slab and a bit (72)."""
    options.set("GEMM_TILE", form)
    W, m, n = 4, 392, 600
    g = torch.Generator().manual_seed(form)
    datas = [(((torch.rand((m, k // W), generator=g) * 2 - 1) * 0.05).to(dtype),
              ((torch.rand((n, k // W), generator=g) * 2 - 1) * 0.05).to(dtype),
              None) for _ in range(W)]
    bias = ((torch.rand((n,), generator=g) * 2 - 1) * 0.05).to(dtype)
    datas = [(x, w, bias) for x, w, _ in datas]
    x, w, b = G.pack_world(datas, gpu_device)
    exact = O.exact_world(datas)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    # ragged shards on the wide tiles: on the zero-padded copy of the operands (with the workspace) and
    # in place (without it: the early-starting last slab of a shard)
    for pad_ragged in (True, False):
        out = G.HipGemmReduceScatter(W, pad_ragged=pad_ragged).forward(x, w, b).cpu()
        err = (out.double() - exact).abs()
        assert bool((err <= exact.abs() * ulp + 1e-6).all()), (pad_ragged, float(err.max()))


@pytest.mark.gpu
@pytest.mark.parametrize("form", [256, 129, 131, 132, 130, 128, 32])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_each_kernel_form_by_whole_lines(gpu_device, options, form, dtype):
    """The same with fourteen slabs to a shard, the last a short one, which tiles of 256 rows request by whole lines."""
    test_each_kernel_form(gpu_device, options, form, dtype, 4 * 840)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 256, 129, 131, 132, 130])
@pytest.mark.parametrize("m,n", [(1200, 4352), (1024, 4872), (1301, 2600), (2304, 2304), (640, 6144), (72, 8192), (2816, 3072)])
def test_every_tile_of_odd_tile_counts(gpu_device, options, form, m, n):
    """Tile counts that the dies' blocks and bands cut unevenly (a last group of less than four columns, a last band that is
    short or empty), as the library multiplies them and in every form on 256 rows or columns: no tile is left out or done
    twice.  f32 sums of 8 x 72 products, rounded once: within 2^-8 of the f32 product and 1e-6."""
    options.set("GEMM_TILE", form)
    W, kl = 8, 72
    g = torch.Generator(device=gpu_device).manual_seed(m + n)
    x = torch.empty(W, m, kl, dtype=torch.bfloat16, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    w = torch.empty(W, n, kl, dtype=torch.bfloat16, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    G.HipGemmReduceScatter(W).forward(x, w, None, out=out)
    want = x.transpose(0, 1).reshape(m, W * kl).float() @ w.transpose(0, 1).reshape(n, W * kl).float().T
    torch.cuda.synchronize()
    assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 1e-6).all())


@pytest.mark.skipif(torch.cuda.is_available(), reason="its operands do not exist: no call may reach a GPU")
@pytest.mark.parametrize("W", [2, 8])
def test_the_room_that_is_asked_for_is_enough(W):
    """No shape is refused with the room that gemm_rs_workspace_used or _bytes tells, none among it (such a shape was, where a plan of
    one group took the place of one that had to have room)."""
    lib, rng = _lib.load(), random.Random(W)
    for i in range(1500):
        m, n = 8 * int(2 ** rng.uniform(0, 10)), 4 * int(2 ** rng.uniform(6, 11.5))
        k = W * 8 * int(2 ** rng.uniform(3, 9))
        for need in (lib.gemm_rs_workspace_used(m, n, k, W), lib.gemm_rs_workspace_bytes(m, n, k, W)):
            rc = lib.gemm_rs_forward(4096, 4096, None, 4096, m, n, k, W, 0, 0, _lib.BF16, 4096 if need else None, need, None)
            assert rc != E_WORKSPACE, (m, n, k)


@pytest.mark.parametrize("W", [2, 8])
def test_the_room_that_is_told_is_enough_on_the_host(W):
    """The same of the entry point compiled for the host, which runs everywhere: nothing is launched."""
    rng, shapes = random.Random(W), []
    for i in range(1500):
        m, n = 8 * int(2 ** rng.uniform(0, 10)), 4 * int(2 ** rng.uniform(6, 11.5))
        shapes.append((m, n, 8 * int(2 ** rng.uniform(3, 9)), W, 0, 0, 0, 0))
    told = [got[-2:] for got in tile_loops.run([("call", 0, 0, *s, 0, 0) for s in shapes])]
    calls = [("call", 0, 0, *s, need, 0) for s, needs in zip(shapes, told) for need in needs]
    for call, got in zip(calls, tile_loops.run(calls)):
        assert got[0] == "0", (call, got)


ROOM_OF_EARLIER = [  # W, m, n, kl, bytes, kernels: what gemm_rs_workspace_bytes has told of for these, and is enough for them
    (16, 153, 10936, 2304, 4 * 153 * 10936 * 4, "split reduce"), (8, 1976, 2304, 3216, 2 * 1976 * 2304 * 4, "split reduce"),
    (8, 1162, 3836, 3720, 2 * 1162 * 3836 * 4, "split reduce"), (8, 35928, 4, 392, 0, "narrow"), (8, 36053, 4, 4960, 0, "narrow"),
]


@pytest.mark.parametrize("W,m,n,kl,room,kernels", ROOM_OF_EARLIER)
def test_room_that_was_enough_is(W, m, n, kl, room, kernels):
    """Calls with less room than the form that is chosen now asks for: answered with as much as they were, and with the first byte of
    it missing, or off its alignment, refused."""
    call = lambda size, at=0: tile_loops.run([("call", 0, 0, m, n, kl, W, 0, 0, 0, 0, size, at)])[0][:-2]
    assert call(room) == ["0", *kernels.split()]
    if room:
        assert call(room - 1) == call(room, 8) == call(0) == [str(E_WORKSPACE)]  # (less than the others have to have)


def launched(lib, call):
    """Names of the kernels that call() launches."""
    assert lib.moe_a2a_timer_begin(8) == 0
    call()
    torch.cuda.synchronize()
    ids, us = (ctypes.c_int * 8)(), (ctypes.c_float * 8)()
    return [lib.moe_a2a_kernel_name(ids[i]).decode() for i in range(lib.moe_a2a_timer_end(ids, us, 8))]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,kernel", [
    (2816, 2944, 2048, "gemm_rs_narrow"),  # 132 wide tiles, but one round of 253 narrow ones
    (4300, 1900, 1088, "gemm_rs_narrow"),  # the same off the grid of 128-byte lines, ragged in both directions
    (1408, 5504, 2048, "gemm_rs_narrow"),  # 132 wide tiles, two rounds of narrow ones with 128 rows in use
    (1408, 5504, 4608, "gemm_rs_wide"),  # the same with a longer K
    (1280, 6656, 2048, "gemm_rs_wide"),  # 130 wide tiles, three rounds of 128 rows
    (264, 16640, 2048, "gemm_rs_wide"),  # few rows
    (2048, 4096, 2048, "gemm_rs_narrow"),  # 128
])
def test_tile_width_where_wide_tiles_begin(gpu_device, m, n, k, kernel):
    """Either side of the rules that choose the tiles, by the kernel that is launched, and its results: f32 sums of k products
    of up to 0.05^2, rounded once, within 2^-8 of the f32 product and 1e-5."""
    W = 8
    g = torch.Generator(device=gpu_device).manual_seed(m + n + k)
    x = torch.empty(W, m, k // W, dtype=torch.bfloat16, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    w = torch.empty(W, n, k // W, dtype=torch.bfloat16, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    assert launched(_lib.load(), lambda: G.HipGemmReduceScatter(W).forward(x, w, None, out=out)) == [kernel]
    want = x.transpose(0, 1).reshape(m, k).float() @ w.transpose(0, 1).reshape(n, k).float().T
    assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 1e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("k,grouped", [(20160, "gemm_rs_split"), (16384, "gemm_rs_narrow")])
def test_partial_products_are_optional_for_many_tiles(gpu_device, k, grouped):
    """185 tiles of 256 x 128 with shards long enough that groups of them pay: the call is accepted without a workspace, with
    one that is too small and with one off its alignment, and then sums all shards in one place.  f32 sums of k products
    of up to 0.05^2, rounded once: within 2^-8 of the f32 product and 2e-5."""
    lib, W, m, n = _lib.load(), 8, 1176, 4672
    g = torch.Generator(device=gpu_device).manual_seed(3)
    x = torch.empty(W, m, k // W, dtype=torch.bfloat16, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    w = torch.empty(W, n, k // W, dtype=torch.bfloat16, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    want = x.transpose(0, 1).reshape(m, k).float() @ w.transpose(0, 1).reshape(n, k).float().T
    need = lib.gemm_rs_workspace_bytes(m, n, k, W)
    assert need >= 2 * m * n * 4
    ws = torch.empty(need + 16, dtype=torch.uint8, device=gpu_device)
    outs = []
    for at, size, kernels in ((None, 0, ["gemm_rs_narrow"]), (ws.data_ptr(), need - 1, ["gemm_rs_narrow"]),
                              (ws.data_ptr() + 8, need, ["gemm_rs_narrow"]),
                              (ws.data_ptr(), need, [grouped, "gemm_rs_reduce"])):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)

        def call():
            assert lib.gemm_rs_forward(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, k, W, 0, 0, _lib.BF16, at, size,
                                       torch.cuda.current_stream().cuda_stream) == 0
        assert launched(lib, call) == kernels
        assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 2e-5).all())
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 33, 64])
@pytest.mark.parametrize("W,n,kl", [
    (1, 8, 64), (1, 200, 192), (8, 8, 64), (2, 72, 128), (3, 200, 256),  # fewer slabs than are kept in flight, ragged columns
    (8, 72, 72), (8, 2880, 360), (2, 4104, 1160), (8, 8200, 456),  # rows that end inside a slab
    (8, 1000, 320), (8, 2880, 384), (4, 4104, 1024), (8, 8200, 512), (8, 32760, 128),  # tiles of 64 columns, of 128, one group
    (1, 200, 200), (8, 32760, 72), (8, 32776, 128),  # one group of rows that end inside a slab; more columns: 256 x 256 tiles
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_few_rows(gpu_device, dtype, m, W, n, kl):
    """The weight-streaming form: every row and column, whatever the tile width and the groups, with a bias.
    f32 sums of W kl products of up to 0.05^2, rounded once: within 2^-8 (fp16: 2^-11) of the f32 result and 1e-5."""
    g = torch.Generator(device=gpu_device).manual_seed(m + n + kl)
    x = torch.empty(W, m, kl, dtype=dtype, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    w = torch.empty(W, n, kl, dtype=dtype, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    bias = torch.empty(n, dtype=dtype, device=gpu_device).uniform_(-0.01, 0.01, generator=g)
    out = torch.full((m, n), float("nan"), dtype=dtype, device=gpu_device)
    kernels = launched(_lib.load(), lambda: G.HipGemmReduceScatter(W).forward(x, w, bias, out=out))
    groups = _lib.load().gemm_rs_workspace_bytes(m, n, W * kl, W) // (4 * m * n)
    assert kernels[0] == ("gemm_rs_tile" if n <= 32768 else "gemm_rs_wide") and kernels[1:] in ([], ["gemm_rs_reduce"])
    assert groups or len(kernels) == 1
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    want = x.transpose(0, 1).reshape(m, W * kl).float() @ w.transpose(0, 1).reshape(n, W * kl).float().T + W * bias.float()
    torch.cuda.synchronize()
    assert bool(((out.float() - want).abs() <= want.abs() * ulp + 1e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 37, 64])
@pytest.mark.parametrize("W,n,kl,at", [
    (8, 8200, 680, 0), (8, 8190, 712, 3),  # rows that start a line every eighth time; operands that start 48 bytes into one
    (8, 8200, 736, 4), (3, 32744, 456, 1),  # on half lines; groups that do not divide the dies
    (1, 32760, 1352, 5), (2, 32766, 696, 0),  # one group; an odd number of results in the last tile
    (8, 7176, 2056, 7),  # more weights than stay in the memory-side cache
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_few_rows_by_whole_lines(gpu_device, dtype, m, W, n, kl, at):
    """Rows off the grid of cache lines and more than 84 MiB of weights: chunks that lag a request behind, at the shards' first and
    last slabs, with an infinite element in either operand's last column.  Shards 24 and 40 elements apart whose gaps hold NaN.
    f32 sums of W kl products of up to 0.05^2, rounded once: within 2^-8 (fp16: 2^-11) of the f32 result and 1e-5."""
    lib, gaps = _lib.load(), (24, 40)
    flat, parts = [], []
    for rows, gap, seed in ((m, gaps[0], 1), (n, gaps[1], 2)):
        t = torch.full((8 * at + W * (rows * kl + gap),), float("nan"), dtype=dtype, device=gpu_device)
        part = t[8 * at:].view(W, rows * kl + gap)[:, :rows * kl].unflatten(1, (rows, kl))
        part.copy_(uniform((W, rows, kl), dtype, gpu_device, seed + kl))
        flat.append(t)
        parts.append(part)
    x, w = parts
    x[W - 1, m - 1, kl - 1] = float("inf")
    w[0, n - 1, kl - 1] = float("-inf")
    w[W - 1, 5, 0] = float("inf")
    out = torch.full((m, n), float("nan"), dtype=dtype, device=gpu_device)
    ws = torch.empty(max(16, lib.gemm_rs_workspace_bytes(m, n, kl * W, W)), dtype=torch.uint8, device=gpu_device)
    assert lib.gemm_rs_forward(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, kl * W, W, m * kl + gaps[0], n * kl + gaps[1],
                               _lib.BF16 if dtype == torch.bfloat16 else _lib.F16, ws.data_ptr(), ws.numel(),
                               torch.cuda.current_stream().cuda_stream) == 0
    want = product(x, w)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    ulp, finite = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11, want.isfinite()
    assert bool(((out.float() - want).abs() <= want.abs() * ulp + 1e-5)[finite].all())


@pytest.mark.gpu
@pytest.mark.parametrize("form,W,m", [(0, 4, 64), (0, 1, 5), (256, 4, 392), (129, 4, 392), (131, 4, 392), (132, 4, 392),
                                      (130, 4, 392), (128, 4, 392), (32, 4, 392)])
@pytest.mark.parametrize("kl", [72, 352, 360, 456])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_non_finite_elements_of_ragged_shards(gpu_device, options, dtype, kl, form, W, m):
    """Infinities and NaN in the columns that a last slab which starts early shares with the one before (and elsewhere), in
    either operand, padded and in place: NaN and infinite of the same sign exactly where the f32 product is, and the other
    results as everywhere (f32 sums rounded once: 2^-8 or 2^-11 of the result, and 1e-6)."""
    options.set("GEMM_TILE", form)
    n, inf, nan = 600, float("inf"), float("nan")
    shared = range(kl - 64, kl // 64 * 64)  # the first and last of these, and a column behind them
    g = torch.Generator(device=gpu_device).manual_seed(kl + form)
    x = torch.empty(W, m, kl, dtype=dtype, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    w = torch.empty(W, n, kl, dtype=dtype, device=gpu_device).uniform_(-0.05, 0.05, generator=g)
    for i, (col, value) in enumerate([(shared[0], inf), (shared[-1], -inf), (shared[0], nan), (kl - 1, inf), (0, -inf)]):
        w[i % W, 7 + 113 * i, col] = value
    x[W - 1, m // 3, shared[-1]] = inf
    x[0, m - 1, shared[0]] = nan
    x[0, 0, shared[0]] = -inf
    want = x.transpose(0, 1).reshape(m, W * kl).float() @ w.transpose(0, 1).reshape(n, W * kl).float().T
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for pad_ragged in (True, False):
        out = G.HipGemmReduceScatter(W, pad_ragged=pad_ragged).forward(x, w).float()
        torch.cuda.synchronize()
        assert torch.equal(out.isnan(), want.isnan()), pad_ragged
        assert torch.equal(out.isposinf(), want.isposinf()) and torch.equal(out.isneginf(), want.isneginf()), pad_ragged
        finite = want.isfinite()
        assert bool(((out - want).abs() <= want.abs() * ulp + 1e-6)[finite].all()), pad_ragged


@pytest.mark.gpu
@pytest.mark.parametrize("form,W,m", [(0, 4, 64), (0, 1, 5), (256, 4, 392), (129, 4, 392), (131, 4, 392), (132, 4, 392),
                                      (130, 4, 392), (128, 4, 392), (32, 4, 392)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_non_finite_elements_of_long_ragged_shards(gpu_device, options, dtype, form, W, m):
    """The same with fourteen slabs to a shard, which tiles of 256 rows request by whole lines."""
    test_non_finite_elements_of_ragged_shards(gpu_device, options, dtype, 840, form, W, m)


@pytest.mark.gpu
def test_local_k_with_a_short_last_slab_and_one_rank(gpu_device):
    """Local K = 360 (five slabs of 64 and one of 40, the reference's 2880 / 8), and a world of one."""
    for W, m, n, k in ((8, 64, 2880, 2880), (1, 130, 136, 72)):
        datas = [G.generate_input(r, W, m if m % W == 0 else m, n, k, True, 5) if m % W == 0 else None for r in range(W)]
        if datas[0] is None:  # M need not divide by W for the sum itself
            g = torch.Generator().manual_seed(9)
            datas = [(((torch.rand((m, k // W), generator=g) * 2 - 1) * 0.01).to(torch.bfloat16),
                      ((torch.rand((n, k // W), generator=g) * 2 - 1) * 0.01).to(torch.bfloat16), None)
                     for _ in range(W)]
        x, w, b = G.pack_world(datas, gpu_device)
        out = G.HipGemmReduceScatter(W).forward(x, w, b).cpu()
        ok, worst = within_one_rounding(out, O.exact_world(datas))
        assert ok, worst


@pytest.mark.gpu
@pytest.mark.parametrize("form", [256, 129, 131, 130, 128, 32])
def test_shards_with_gaps_between_them(gpu_device, options, form):
    """Shard strides of the C ABI: the shards of each operand lie further apart than their size."""
    options.set("GEMM_TILE", form)
    lib = _lib.load()
    W, m, n, kl, gap_a, gap_b = 4, 264, 272, 128, 64, 200
    g = torch.Generator().manual_seed(31)
    datas = [(((torch.rand((m, kl), generator=g) * 2 - 1) * 0.05).to(torch.bfloat16),
              ((torch.rand((n, kl), generator=g) * 2 - 1) * 0.05).to(torch.bfloat16), None) for _ in range(W)]
    sa, sb = m * kl + gap_a, n * kl + gap_b
    a = torch.full((W * sa,), float("nan"), dtype=torch.bfloat16, device=gpu_device)  # the gaps hold NaN
    b = torch.full((W * sb,), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    for s, (x, w, _) in enumerate(datas):
        a[s * sa:s * sa + m * kl] = x.to(gpu_device).reshape(-1)
        b[s * sb:s * sb + n * kl] = w.to(gpu_device).reshape(-1)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu_device)
    need = int(lib.gemm_rs_workspace_bytes(m, n, kl * W, W))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=gpu_device)
    rc = lib.gemm_rs_forward(a.data_ptr(), b.data_ptr(), None, out.data_ptr(), m, n, kl * W, W, sa, sb, _lib.BF16,
                             ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    ok, worst = within_one_rounding(out.cpu(), O.exact_world(datas))
    assert ok, worst


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8, 64, 512, 8 * 256), (4, 520, 520, 4 * 128)], ids=["partial-products", "tiles"])
def test_replays_of_a_captured_graph_follow_their_inputs(gpu_device, shape):
    """The entry point only enqueues kernels (the grouped form: the tile kernel, then the reduction
    over its partial products in the caller's workspace), so a call can be captured into a hipGraph;
    every replay is checked against an eager run on the inputs of the moment, with eager work and
    synchronisations between the replays."""
    W, m, n, k = shape
    op = G.HipGemmReduceScatter(W)
    g = torch.Generator().manual_seed(77)
    fresh = lambda: (((torch.rand((W, m, k // W), generator=g) * 2 - 1) * 0.05).to(torch.bfloat16).to(gpu_device),
                     ((torch.rand((W, n, k // W), generator=g) * 2 - 1) * 0.05).to(torch.bfloat16).to(gpu_device),
                     ((torch.rand((n,), generator=g) * 2 - 1) * 0.05).to(torch.bfloat16).to(gpu_device))
    x, w, b = fresh()
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu_device)
    op.forward(x, w, b, out=out)  # allocates the workspace outside the capture
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            op.forward(x, w, b, out=out)
    for _ in range(3):
        nx, nw, nb = fresh()
        x.copy_(nx), w.copy_(nw), b.copy_(nb)
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        eager = G.HipGemmReduceScatter(W).forward(x, w, b)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), eager.view(torch.int16))
        ok, worst = within_one_rounding(got.cpu(), O.exact_world([(x[s].cpu(), w[s].cpu(), b.cpu()) for s in range(W)]))
        assert ok, worst


def product(x, w, bias=None):
    """The f32 product of concatenated shards."""
    W, m, kl = x.shape
    y = x.transpose(0, 1).reshape(m, W * kl).float() @ w.transpose(0, 1).reshape(w.shape[1], W * kl).float().T
    return y if bias is None else y + W * bias.float()


def uniform(shape, dtype, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.empty(*shape, dtype=dtype, device=dev).uniform_(-0.05, 0.05, generator=g)


@pytest.mark.gpu
@pytest.mark.parametrize("W,m,n,kl", [
    (2, 65, 8, 64), (2, 256, 256, 72), (8, 257, 260, 64), (4, 392, 600, 360), (8, 72, 4100, 96), (3, 520, 2052, 200),
    (4, 1040, 1000, 128),  # more than a round of tiles
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_wide_tiles_with_the_shards_in_groups(gpu_device, options, dtype, W, m, n, kl):
    """Every row and column at the edges of tiles, slabs and groups, with a bias and an infinite element on either side.  f32
    sums of W kl products of up to 0.05^2, rounded once: within 2^-8 (fp16: 2^-11) of the f32 product and 1e-5."""
    options.set("GEMM_TILE", 133)
    x, w, bias = (uniform(s, dtype, gpu_device, m + n + i) for i, s in enumerate(((W, m, kl), (W, n, kl), (n,))))
    x[W - 1, m - 1, kl - 1] = float("inf")
    w[0, n - 1, kl - 8] = float("-inf")
    out = torch.full((m, n), float("nan"), dtype=dtype, device=gpu_device)
    kernels = launched(_lib.load(), lambda: G.HipGemmReduceScatter(W).forward(x, w, bias, out=out))
    assert kernels == ["gemm_rs_split", "gemm_rs_reduce"]
    want = product(x, w, bias)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    ulp, finite = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11, want.isfinite()
    assert bool(((out.float() - want).abs() <= want.abs() * ulp + 1e-5)[finite].all())


@pytest.mark.gpu
@pytest.mark.parametrize("form,W,m,n,kl,at", [
    (256, 8, 2056, 264, 712, 0), (256, 3, 1030, 520, 728, 3), (256, 2, 520, 260, 1000, 5),  # rows alike eight, four apart, too few
    (256, 1, 300, 256, 904, 7), (256, 2, 4104, 72, 720, 1), (256, 4, 1291, 40, 744, 2),  # one shard; half lines; classes of unequal length
    (133, 8, 1030, 264, 72, 3), (133, 2, 1040, 260, 136, 5), (133, 4, 530, 520, 200, 6), (133, 2, 257, 256, 264, 1),  # two slabs, three, four, five
    (129, 4, 520, 264, 136, 3), (131, 3, 400, 264, 200, 6), (132, 2, 264, 520, 72, 1), (130, 4, 300, 264, 456, 7),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_tiles_by_whole_lines(gpu_device, options, dtype, form, W, m, n, kl, at):
    """Rows off the grid of cache lines on the tiles of eight waves: chunks that lag a request behind, at the first and last slabs of
    shards and past the last one, rows of x that lie alike dealt to the same tile, with an infinite element in either operand's last column
    and its first.  Operands that start 16 `at` bytes into a line, and shards 24 and 40 elements apart whose gaps hold NaN.  f32 sums
    of W kl products of up to 0.05^2, rounded once: within 2^-8 (fp16: 2^-11) of the f32 result and 1e-5."""
    lib, gaps = _lib.load(), (24, 40)
    options.set("GEMM_TILE", form)
    flat, parts = [], []
    for rows, gap, seed in ((m, gaps[0], 1), (n, gaps[1], 2)):
        t = torch.full((8 * at + W * (rows * kl + gap),), float("nan"), dtype=dtype, device=gpu_device)
        part = t[8 * at:].view(W, rows * kl + gap)[:, :rows * kl].unflatten(1, (rows, kl))
        part.copy_(uniform((W, rows, kl), dtype, gpu_device, seed + kl))
        flat.append(t)
        parts.append(part)
    x, w = parts
    x[W - 1, m - 1, kl - 1] = float("inf")
    x[0, m // 2, 0] = float("-inf")
    w[0, n - 1, kl - 1] = float("-inf")
    w[W - 1, 5, 0] = float("inf")
    out = torch.full((m, n), float("nan"), dtype=dtype, device=gpu_device)
    ws = torch.empty(max(16, lib.gemm_rs_workspace_bytes(m, n, kl * W, W)), dtype=torch.uint8, device=gpu_device)
    assert lib.gemm_rs_forward(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, kl * W, W, m * kl + gaps[0], n * kl + gaps[1],
                               _lib.BF16 if dtype == torch.bfloat16 else _lib.F16, ws.data_ptr(), ws.numel(),
                               torch.cuda.current_stream().cuda_stream) == 0
    want = product(x, w)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    ulp, finite = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11, want.isfinite()
    assert bool(((out.float() - want).abs() <= want.abs() * ulp + 1e-5)[finite].all())


def check_off_the_line_grid(dev, dtype, W, m, n, kl, at, gaps=(24, 40)):
    """The product of shards whose rows lie off the grid of cache lines, with an infinite element in either operand's last column and its
    first.  Operands that start 16 `at` bytes into a line, and shards so many elements apart whose gaps hold NaN.  f32 sums of W kl
    products of up to 0.05^2, rounded once: within 2^-8 (fp16: 2^-11) of the f32 result and 1e-5.  The kernels that ran."""
    lib = _lib.load()
    flat, parts = [], []
    for rows, gap, seed in ((m, gaps[0], 1), (n, gaps[1], 2)):
        t = torch.full((8 * at + W * (rows * kl + gap),), float("nan"), dtype=dtype, device=dev)
        part = t[8 * at:].view(W, rows * kl + gap)[:, :rows * kl].unflatten(1, (rows, kl))
        part.copy_(uniform((W, rows, kl), dtype, dev, seed + kl))
        flat.append(t)
        parts.append(part)
    x, w = parts
    x[W - 1, m - 1, kl - 1] = float("inf")
    x[0, m // 2, 0] = float("-inf")
    w[0, n - 1, kl - 1] = float("-inf")
    w[W - 1, 5, 0] = float("inf")
    out = torch.full((m, n), float("nan"), dtype=dtype, device=dev)
    ws = torch.empty(max(16, lib.gemm_rs_workspace_bytes(m, n, kl * W, W)), dtype=torch.uint8, device=dev)
    rc = []
    kernels = launched(lib, lambda: rc.append(lib.gemm_rs_forward(
        x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, kl * W, W, m * kl + gaps[0], n * kl + gaps[1],
        _lib.BF16 if dtype == torch.bfloat16 else _lib.F16, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)))
    assert rc == [0]
    want = product(x, w)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    ulp, finite = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11, want.isfinite()
    assert bool(((out.float() - want).abs() <= want.abs() * ulp + 1e-5)[finite].all())
    return kernels


@pytest.mark.gpu
@pytest.mark.parametrize("form,W,m,n,kl,at", [
    (256, 2, 6160, 6144, 72, 3), (256, 1, 6144, 6152, 136, 5), (256, 2, 6150, 6144, 200, 6), (256, 1, 6152, 6144, 264, 1),  # two slabs, three, four, five
    (133, 8, 2060, 1032, 72, 3), (133, 8, 2060, 1032, 136, 5), (133, 4, 4120, 1032, 200, 6), (133, 8, 2060, 1032, 264, 1),
    (133, 8, 1030, 264, 584, 3), (133, 2, 1040, 260, 648, 5), (133, 4, 530, 520, 712, 6), (133, 2, 257, 256, 776, 1),
    (129, 4, 520, 264, 776, 3),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_tiles_by_whole_lines_from_where_these_begin(gpu_device, options, dtype, form, W, m, n, kl, at):
    """The same where whole lines are chosen on both sides of gemm_rs_along: short shards of large outputs or of more tiles than a round of the
    CUs, and long ones (check_off_the_line_grid)."""
    options.set("GEMM_TILE", form)
    check_off_the_line_grid(gpu_device, dtype, W, m, n, kl, at)


@pytest.mark.gpu
@pytest.mark.parametrize("form,W,m,n,kl,at", [
    (129, 2, 2304, 2570, 72, 3), (129, 3, 2312, 2440, 200, 5), (129, 1, 2305, 2432, 680, 1), (129, 8, 2296, 2561, 96, 4),
    (133, 8, 1030, 264, 72, 3), (133, 2, 1040, 260, 136, 5), (133, 4, 530, 520, 200, 6), (133, 2, 257, 256, 264, 1), (129, 4, 520, 264, 136, 3),
    (129, 2, 300, 200, 160, 2), (131, 4, 400, 264, 224, 4), (132, 3, 264, 520, 416, 0), (130, 8, 520, 264, 96, 6), (130, 2, 300, 132, 352, 5),  # half lines
    (133, 8, 1030, 264, 96, 3), (133, 2, 257, 256, 672, 1), (133, 4, 530, 520, 736, 6), (133, 2, 1000, 264, 1184, 2),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_tiles_of_rows_as_they_lie(gpu_device, options, dtype, form, W, m, n, kl, at):
    """Short shards off the grid of cache lines, which 256 x 128 tiles with all rows in use and 256 x 256 tiles in groups request as they lie,
    and shards on half lines, where the other 256 x 128 tiles do (check_off_the_line_grid)."""
    options.set("GEMM_TILE", form)
    check_off_the_line_grid(gpu_device, dtype, W, m, n, kl, at)


@pytest.mark.gpu
@pytest.mark.parametrize("kl", [256, 96, 136, 360, 776, 840])
def test_same_bits(gpu_device, options, kl):
    """What include/gemm_rs.h says of the order of sums: the same in all unsplit forms, but for 256 x 256 tiles off the grid of 64, and the same
    wherever the operands begin, but for these tiles by whole lines (from twelve slabs on, here)."""
    W, m, n, results = 4, 392, 600, {}
    for at in (0, 24, 40):  # elements: on the grid of cache lines, and 48 and 80 bytes off it
        x, w = (torch.empty(8 * 8 + W * r * kl, dtype=torch.bfloat16, device=gpu_device)[at:at + W * r * kl].view(W, r, kl) for r in (m, n))
        x.copy_(uniform((W, m, kl), torch.bfloat16, gpu_device, kl))
        w.copy_(uniform((W, n, kl), torch.bfloat16, gpu_device, kl + 1))
        for form in (129, 131, 132, 128, 256):
            options.set("GEMM_TILE", form)
            out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
            G.HipGemmReduceScatter(W).forward(x, w, out=out)
            results[form, at] = out.view(torch.int16)
    for (form, at), got in results.items():
        if form != 256 or kl % 64 == 0:
            assert torch.equal(got, results[129, 0]), (form, at)
        elif kl <= 11 * 64:
            assert torch.equal(got, results[256, 0]), at


@pytest.mark.gpu
@pytest.mark.parametrize("form,m,n,kl,kernels", [
    (256, 520, 264, 776, "wide"), (133, 520, 264, 776, "split reduce"), (129, 520, 264, 776, "narrow"), (131, 400, 264, 360, "narrow"),
    (132, 300, 264, 200, "narrow"), (130, 300, 264, 456, "narrow reduce"), (0, 40, 8200, 2728, "tile reduce"),  # (more than 84 MiB of weights)
])
def test_shards_far_apart(gpu_device, options, form, m, n, kl, kernels):
    """Two shards of either operand, more than a 32-bit offset apart (2 GiB): the same form as of shards that are near, and rows as they lie
    (check_off_the_line_grid)."""
    options.set("GEMM_TILE", form)
    assert check_off_the_line_grid(gpu_device, torch.bfloat16, 2, m, n, kl, 3, ((1 << 30) + 24, (1 << 30) + 40)) == ["gemm_rs_" + k for k in kernels.split()]


@pytest.mark.gpu
@pytest.mark.parametrize("form,W,m,n,kl", [
    (0, 8, 128, 1, 360), (0, 2, 65, 1, 72), (0, 8, 1, 32776, 720), (0, 1, 1, 33000, 712),
    (256, 8, 1, 300, 712), (256, 8, 300, 1, 712), (256, 1, 1, 1, 776), (129, 8, 1, 300, 72), (129, 2, 300, 1, 104), (129, 8, 1, 300, 776), (129, 2, 300, 1, 712), (131, 3, 1, 200, 360),
    (131, 8, 200, 1, 200), (132, 8, 1, 140, 456), (132, 1, 70, 1, 80), (130, 8, 1, 140, 72), (133, 8, 1, 300, 712), (133, 2, 1, 4, 136),
])
def test_operands_of_one_row(gpu_device, options, form, W, m, n, kl):
    """Rows off the grid of cache lines whose shards begin less than a line behind the last one's end (test_tile_loop_addresses.py: every
    request inside the operands).  f32 sums of W kl products of up to 0.05^2, rounded once: within 2^-8 of the f32 result and 1e-5."""
    options.set("GEMM_TILE", form)
    x, w, bias = (uniform(s, torch.bfloat16, gpu_device, m + n + i) for i, s in enumerate(((W, m, kl), (W, n, kl), (n,))))
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    G.HipGemmReduceScatter(W).forward(x, w, bias, out=out)
    want = product(x, w, bias)
    assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 1e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("W,m,n,k,groups,narrow", [(8, 512, 5440, 17024, 4, "groups"), (8, 240, 4480, 24128, 8, "groups"),
                                                   (8, 1096, 6400, 6464, 2, "whole"), (4, 304, 5696, 11328, 4, "groups"),
                                                   (8, 120, 4160, 11008, 8, "groups")])
def test_room_for_the_groups_is_optional(gpu_device, options, W, m, n, k, groups, narrow):
    """Shapes that take 256 x 256 tiles in groups: room for their partial products is what is asked for, and with less of it, or off its
    alignment, the call is answered as it is without that form: on the 256 x 128 tiles, in fewer groups, which have to have room (or
    MOE_A2A_E_WORKSPACE, MOE_A2A_E_ALIGN), or, where these give most CUs a tile (250 of them), whole, with no room at all and
    the bits of that form.  Shards that lie apart as well.  Tolerance as above, 2e-5."""
    lib = _lib.load()
    pad = 64
    x, w = uniform((W, m * (k // W) + pad), torch.bfloat16, gpu_device, 5), uniform((W, n * (k // W) + pad), torch.bfloat16, gpu_device, 6)
    want = product(x[:, :-pad].reshape(W, m, -1), w[:, :-pad].reshape(W, n, -1))
    need = lib.gemm_rs_workspace_bytes(m, n, k, W)
    assert need == groups * m * n * 4
    ws = torch.empty(need + 16, dtype=torch.uint8, device=gpu_device)

    def call(at, size):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
        rc = []
        kernels = launched(lib, lambda: rc.append(lib.gemm_rs_forward(
            x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, k, W, m * (k // W) + pad, n * (k // W) + pad, _lib.BF16, at, size,
            torch.cuda.current_stream().cuda_stream)))
        assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 2e-5).all()) if rc == [0] else bool(out.isnan().all())
        return rc + kernels, out

    assert call(ws.data_ptr(), need)[0] == [0, "gemm_rs_split", "gemm_rs_reduce"]
    less = (ws.data_ptr(), need - 1), (ws.data_ptr() + 8, need), (None, 0)
    if narrow == "groups":
        assert [call(*room)[0] for room in less] == [[0, "gemm_rs_narrow", "gemm_rs_reduce"], [E_ALIGN], [E_WORKSPACE]]
    else:
        got = [call(*room) for room in less]
        options.set("GEMM_TILE", 129)
        got.append(call(None, 0))
        assert all(how == [0, "gemm_rs_narrow"] and torch.equal(out, got[0][1]) for how, out in got)


@pytest.mark.gpu
@pytest.mark.parametrize("W,m,n,kl,room,kernels", ROOM_OF_EARLIER)
def test_results_with_room_that_was_enough(gpu_device, W, m, n, kl, room, kernels):
    """f32 sums of W kl products of up to 0.05^2, rounded once: within 2^-8 of the f32 result and 2e-5."""
    lib = _lib.load()
    x, w = uniform((W, m, kl), torch.bfloat16, gpu_device, m), uniform((W, n, kl), torch.bfloat16, gpu_device, n)
    out, ws = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device), torch.empty(max(room, 16), dtype=torch.uint8, device=gpu_device)
    rc = []
    names = launched(lib, lambda: rc.append(lib.gemm_rs_forward(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, W * kl, W, 0, 0, _lib.BF16,
                                                                ws.data_ptr() if room else None, room, torch.cuda.current_stream().cuda_stream)))
    assert rc == [0] and names == ["gemm_rs_" + k for k in kernels.split()]
    want = product(x, w)
    assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 2e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(2304, 6656), (2200, 6500), (6736, 2240), (3576, 4416), (7288, 4160)])
def test_wide_tiles_dealt_out_in_column_order(gpu_device, m, n):
    """Numbers of 256 x 256 tiles that bands or blocks would make more rounds of: none left out or done twice."""
    x, w = uniform((8, m, 72), torch.bfloat16, gpu_device, m), uniform((8, n, 72), torch.bfloat16, gpu_device, n)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    assert launched(_lib.load(), lambda: G.HipGemmReduceScatter(8).forward(x, w, out=out)) == ["gemm_rs_wide"]
    want = product(x, w)
    assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 1e-6).all())


@pytest.mark.gpu
def test_workspace_of_a_stream_and_of_a_graph(gpu_device):
    """Calls on two streams at once do not share their partial products, and a captured graph has room of its own, which the handle's
    later calls, or its end, do not take away.  A kept workspace belongs to one stream and is found again; four are kept."""
    W, m, n, k = 8, 1096, 6400, 6464
    h = G.HipGemmReduceScatter(W)
    streams = [torch.cuda.Stream() for _ in range(6)]

    def room(stream):
        with torch.cuda.stream(stream):
            return h.workspace_for(m, n, k, gpu_device)

    a, b = room(streams[0]), room(streams[1])
    assert a.data_ptr() != b.data_ptr() and room(streams[0]) is a and room(streams[1]) is b
    with torch.cuda.stream(streams[1]):
        assert h.workspace_for(64, 256, 1024, gpu_device) is b  # (a smaller one)
    graph, held = torch.cuda.CUDAGraph(), []
    x, w = uniform((W, m, k // W), torch.bfloat16, gpu_device, 1), uniform((W, n, k // W), torch.bfloat16, gpu_device, 2)
    out = torch.empty(m, n, dtype=torch.bfloat16, device=gpu_device)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=streams[0]):
        held.append(h.workspace_for(m, n, k, gpu_device).data_ptr())
        h.forward(x, w, out=out)
    assert held[0] not in (a.data_ptr(), b.data_ptr()) and room(streams[0]) is a
    for s in streams:
        room(s)
    assert len(h._workspaces) == h.MAX_WORKSPACES and room(streams[5]) is room(streams[5])
    del h, a, b
    other = [torch.full((need,), 7, dtype=torch.uint8, device=gpu_device) for need in [2 * m * n * 4] * 8]  # whatever was given back
    want = product(x, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 2e-5).all())
        assert all(bool((o == 7).all()) for o in other)


@pytest.mark.gpu
@pytest.mark.parametrize("kl", [64, 200, 576, 776])  # whole slabs; rows as they lie; whole slabs; whole lines
@pytest.mark.parametrize("m,n", [(2818, 3300), (1500, 7170), (7248, 2304), (868, 8400), (2304, 3700)])
def test_wide_tiles_of_fewer_rows(gpu_device, m, n, kl):
    """Outputs of more than 128 tiles of 256 x 256 that tiles with 192 or 128 of their rows in use cover in as many rounds of the CUs:
    every row and column, a tile's last and the last tile's, with a bias.
    f32 sums of 8 kl products of up to 0.05^2, rounded once: within 2^-8 of the f32 result and 2e-5."""
    x, w = uniform((8, m, kl), torch.bfloat16, gpu_device, m + kl), uniform((8, n, kl), torch.bfloat16, gpu_device, n)
    bias = uniform((n,), torch.bfloat16, gpu_device, 3)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    G.HipGemmReduceScatter(8).forward(x, w, bias, out=out)
    want = product(x, w, bias)
    assert bool(((out.float() - want).abs() <= want.abs() * 2 ** -8 + 2e-5).all())


FEWER_ROWS = [(m, n, kl, rows) for m, n, rows in ((2818, 3300, 192), (1500, 7170, 192), (868, 8400, 128), (2304, 3700, 192))
              for kl in (64, 200, 576, 776)]  # whole slabs; rows as they lie; whole slabs; whole lines
FEWER_ROWS += [(7248, 2304, kl, 192) for kl in (64, 576, 776)]


@pytest.mark.parametrize("m,n,kl,rows", FEWER_ROWS)
def test_rows_in_use_of_wide_tiles(m, n, kl, rows):
    """(tiles down, tiles across, rows in use, how they are dealt to the dies)"""
    kernel, _, _, in_use, _ = tile_loops.run([("call", 2, 0, m, n, kl, 8, 0, 0, 0, 0, 0, 0)])[0][1].split(",")
    assert (kernel, int(in_use)) == ("wide", rows)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,kl,rows", [shape for shape in FEWER_ROWS if shape[:2] in ((2818, 3300), (868, 8400))])
def test_wide_tiles_are_what_runs(gpu_device, m, n, kl, rows):
    """(test_wide_tiles_of_fewer_rows has the results)"""
    x, w = uniform((8, m, kl), torch.bfloat16, gpu_device, m + kl), uniform((8, n, kl), torch.bfloat16, gpu_device, n)
    assert launched(_lib.load(), lambda: G.HipGemmReduceScatter(8).forward(x, w)) == ["gemm_rs_wide"]
