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
