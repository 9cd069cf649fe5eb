"""The forms that fold a token's weighted sum out of registers, at the edges of their dispatch rules: against
the oracle where it is quick, else against the form that reads the dispatched rows back."""
import pytest
import torch

from kernel_amd import contract as C
from kernel_amd.all2all import HipAllToAll
from oracle import all2all_vec as V

pytestmark = pytest.mark.gpu


def bits(t):
    return t.view(torch.int16) if t.dtype in (torch.float16, torch.bfloat16) else t


def inputs(E, K, H, T, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    idx = torch.rand(T, E, generator=g).topk(K, 1).indices.to(torch.int32)
    idx[T // 2] = idx[T // 2, 0]  # one token that names one expert K times
    return torch.randn(T, H, generator=g).to(dtype), idx.contiguous(), torch.rand(T, K, generator=g)


@pytest.mark.parametrize("E,K,H,T,fp8", [
    (1024, 3, 256, 70, True),    # more experts than the workgroup of 512 lanes has threads
    (16, 8, 128, 1024, True),    # the largest table of the one-launch fp8 form
    (16, 8, 128, 1025, True),    # ... and the first beyond it
    (64, 1, 256, 257, "pow2"),   # two tokens per tile
    (32, 32, 384, 5, True),
    (1024, 2, 64, 300, False),
    (12, 5, 2880, 333, False),
    (256, 8, 64, 1100, False),   # tiles of many short tokens
])
@pytest.mark.parametrize("mode", [C.COMBINE_STRICT, C.COMBINE_F32], ids=["strict", "f32"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_fold_equals_the_oracle(gpu_device, E, K, H, T, fp8, mode, dtype):
    cfg = C.MoEConfig(E, K, H, T + 1, dtype, dtype)
    x, idx, w = inputs(E, K, H, T, dtype, E + T)
    want = V.run_world(cfg, [C.RankData(T, idx, w, x)], stub_kind=C.STUB_EXPERT_FRACTION, combine_mode=mode,
                       fp8=bool(fp8), pow2=fp8 == "pow2")
    ata = HipAllToAll(cfg, 0, 1, stub_kind=C.STUB_EXPERT_FRACTION, combine_mode=mode, fp8_dispatch=fp8, fuse_stub=True)
    x, idx, w = x.to(gpu_device), idx.to(gpu_device), w.to(gpu_device)
    for _ in range(2):
        y = ata.forward(x, idx, w)
    torch.cuda.synchronize()
    d = ata.last
    for key in ("counts", "offsets", "slot_of_entry", "src_of_slot", "meta", "disp_x") + (("disp_scale",) if fp8 else ()):
        assert torch.equal(bits(getattr(d, key).cpu()), bits(want[key])), key
    assert torch.equal(bits(y.cpu()), bits(want["y"]))


@pytest.mark.parametrize("T", [5266, 5268])  # x just below and above 72 MB: the cache policy of the rows changes there
@pytest.mark.parametrize("fp8", [False, True])
def test_fold_equals_the_rows_read_back_at_large_x(gpu_device, options, T, fp8):
    E, K, H = 32, 8, 7168
    cfg = C.MoEConfig(E, K, H, T + 1, torch.bfloat16, torch.bfloat16)
    g = torch.Generator(device=gpu_device).manual_seed(T)
    x = torch.randn(T, H, device=gpu_device, generator=g).to(torch.bfloat16)
    idx = torch.rand(T, E, device=gpu_device, generator=g).topk(K, 1).indices.to(torch.int32).contiguous()
    w = torch.rand(T, K, device=gpu_device, generator=g)
    got = []
    for two in (1, 0):
        options.set("TWO_LAUNCHES", two)
        ata = HipAllToAll(cfg, 0, 8, fp8_dispatch=fp8, fuse_stub=True)
        y = ata.forward(x, idx, w)
        got.append((y, ata.last.disp_x, ata.last.slot_of_entry, ata.last.meta))
    for a, b in zip(*got):
        assert torch.equal(bits(a), bits(b))


def same_values(got, want):
    """NaN where the other has NaN (whatever its payload), the same bits elsewhere."""
    got, want = got.cpu(), want.cpu()
    if not got.is_floating_point():
        return torch.equal(got, want)
    return torch.equal(got.isnan(), want.isnan()) and torch.equal(bits(got.nan_to_num()), bits(want.nan_to_num())) \
        and torch.equal(got.isinf(), want.isinf())


def with_specials(x, w):
    """Infinities of both signs, NaN, the largest and the smallest finite values, zeros of both signs in the rows; zero,
    tiny and huge weights."""
    top = torch.finfo(x.dtype).max
    values = torch.tensor([float("inf"), float("-inf"), float("nan"), top, -top, torch.finfo(x.dtype).tiny, 0.0, -0.0])
    T, H = x.shape
    at = torch.arange(T * H).view(T, H)
    x = torch.where(at % 11 == 3, values[at // 11 % 8].to(x.dtype), x)
    w = w.clone()
    w[::3, 0], w[1::5, -1], w[2::7, 0] = 0.0, 1e-30, 3e38
    return x.contiguous(), w


@pytest.mark.parametrize("E,K,H,T", [
    (16, 2, 512, 7),        # a workgroup per token
    (256, 8, 1024, 33),
    (64, 6, 384, 1003),     # a tile of tokens per workgroup
    (12, 5, 64, 500),
    (32, 4, 2048, 9000),    # routed by launches of their own, more rows than the caches hold
])
@pytest.mark.parametrize("mode", [C.COMBINE_STRICT, C.COMBINE_F32], ids=["strict", "f32"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_infinities_and_nan_through_the_fold(gpu_device, E, K, H, T, mode, dtype):
    cfg = C.MoEConfig(E, K, H, T + 1, dtype, dtype)
    x, idx, w = inputs(E, K, H, T, dtype, E + T)
    x, w = with_specials(x, w)
    want = V.run_world(cfg, [C.RankData(T, idx, w, x)], stub_kind=C.STUB_EXPERT_FRACTION, combine_mode=mode)
    ata = HipAllToAll(cfg, 0, 1, stub_kind=C.STUB_EXPERT_FRACTION, combine_mode=mode, fuse_stub=True)
    y = ata.forward(x.to(gpu_device), idx.to(gpu_device), w.to(gpu_device))
    torch.cuda.synchronize()
    assert torch.equal(bits(ata.last.disp_x.cpu()), bits(want["disp_x"]))  # rows are copied, whatever they hold
    assert same_values(y, want["y"])


@pytest.mark.parametrize("E,K,H,T", [(16, 2, 512, 7), (64, 6, 384, 1003), (32, 4, 2048, 9000)])
@pytest.mark.parametrize("fp8", [True, "pow2"])
def test_infinities_and_nan_through_the_fp8_fold(gpu_device, options, E, K, H, T, fp8):
    """Against the form that reads the quantised rows back."""
    cfg = C.MoEConfig(E, K, H, T + 1, torch.bfloat16, torch.bfloat16)
    x, idx, w = inputs(E, K, H, T, torch.bfloat16, E + T)
    x, w = (t.to(gpu_device) for t in with_specials(x, w))
    idx, got = idx.to(gpu_device), []
    for two in (1, 0):
        options.set("TWO_LAUNCHES", two)
        ata = HipAllToAll(cfg, 0, 1, stub_kind=C.STUB_EXPERT_FRACTION, fp8_dispatch=fp8, fuse_stub=True)
        y = ata.forward(x, idx, w)
        got.append((y, ata.last.disp_x, ata.last.disp_scale, ata.last.slot_of_entry, ata.last.meta))
    torch.cuda.synchronize()
    assert all(same_values(a, b) for a, b in zip(*got))
