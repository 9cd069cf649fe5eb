"""The native side of custom_kernel and forward: what it takes over, what it leaves to the long way."""
import copy

import pytest
import torch

from kernel_amd import contract as C
from kernel_amd.all2all import HipAllToAll
from kernel_amd.submission import custom_kernel
from oracle import all2all_vec as V

pytestmark = pytest.mark.gpu


def case(rank, T, dtype=torch.bfloat16, E=16, K=2, H=256):
    g = torch.Generator().manual_seed(100 * rank + T)
    cfg = C.MoEConfig(E, K, H, 64, dtype, dtype)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).to(torch.int32)
    rd = C.RankData(T, idx, torch.rand(T, K, generator=g), torch.randn(T, H, generator=g).to(dtype))
    want = V.run_world(cfg, C.world_of_single_rank(cfg, rd, rank, 8), stub_kind=C.STUB_OWNER_RANK)["y"]
    return cfg, rd.to("cuda:0"), rank, want


def same(y, want):
    return torch.equal(y.cpu().view(torch.int16), want.view(torch.int16))


def test_more_configurations_in_turn_than_are_remembered(gpu_device):
    cases = [case(r, T, dt) for r in range(8) for T in (5, 9) for dt in (torch.bfloat16, torch.float16)]  # 16 keys, two shapes each
    for _ in range(3):
        for cfg, rd, rank, want in cases:
            assert same(custom_kernel((copy.copy(cfg), rd, rank, 8)), want)
    one = cases[0]
    ys = [custom_kernel((one[0], one[1], one[2], 8)) for _ in range(5)]
    assert len({y.data_ptr() for y in ys}) == 5 and all(same(y, one[3]) for y in ys)  # every result is the caller's own


def test_what_the_short_way_does_not_take(gpu_device):
    cfg, rd, rank, want = case(3, 12)
    for _ in range(2):
        assert same(custom_kernel((cfg, rd, rank, 8)), want)
    part = C.RankData(7, rd.indices, rd.weights, rd.x)  # fewer tokens asked for than there are rows
    assert same(custom_kernel((cfg, part, rank, 8)), want[:7])
    strided = C.RankData(12, rd.indices, rd.weights, torch.cat([rd.x, rd.x], 1)[:, : rd.x.shape[1]])
    assert not strided.x.is_contiguous() and same(custom_kernel((cfg, strided, rank, 8)), want)
    for bad in (C.RankData(12, rd.indices.long(), rd.weights, rd.x), C.RankData(12, rd.indices, rd.weights.double(), rd.x),
                C.RankData(12, rd.indices[:, :1].contiguous(), rd.weights, rd.x)):
        with pytest.raises(ValueError):
            custom_kernel((cfg, bad, rank, 8))
    with pytest.raises(RuntimeError):
        custom_kernel((cfg, C.RankData(12, rd.indices.cpu(), rd.weights, rd.x), rank, 8))
    assert same(custom_kernel((cfg, rd, rank, 8)), want)
    changed = copy.copy(cfg)
    custom_kernel((changed, rd, rank, 8))
    changed.experts_per_token = 1  # in place, between two calls
    with pytest.raises(ValueError):
        custom_kernel((changed, rd, rank, 8))


def test_switches_streams_and_phases_between_forwards(gpu_device):
    cfg, rd, rank, _ = case(0, 20)
    ata = HipAllToAll(cfg, 0, 8, fuse_stub=True)
    cpu = rd.to("cpu")
    want = {(s, m): V.run_world(cfg, C.world_of_single_rank(cfg, cpu, 0, 8), stub_kind=s, combine_mode=m)["y"]
            for s in (C.STUB_OWNER_RANK, C.STUB_EXPERT_FRACTION) for m in (C.COMBINE_STRICT, C.COMBINE_F32)}
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(2):
        for (s, m), y in want.items():
            ata.stub_kind, ata.combine_mode = s, m
            assert same(ata.forward(rd.x, rd.indices, rd.weights), y)
            d = ata.dispatch(rd.x, rd.indices)  # flips the sets, in between
            assert d.disp_x.data_ptr() != ata.last.disp_x.data_ptr()
            with torch.cuda.stream(side):
                got = ata.forward(rd.x, rd.indices, rd.weights)
            side.synchronize()
            assert same(got, y) and ata.last.disp_x.data_ptr() != d.disp_x.data_ptr()
    bad = rd.indices.clone()
    bad[4, 1] = cfg.num_experts
    with pytest.raises(IndexError):
        ata.forward(rd.x, bad, rd.weights, check_status=True)
    assert ata.forward(rd.x[:6], rd.indices[:6], rd.weights[:6]).shape[0] == 6


def test_token_counts_in_turn_take_the_short_way(gpu_device, monkeypatch):
    """A call whose token count is not the last one's, but an earlier one's, builds nothing anew: not an argument block,
    not a record; also behind a dispatch of the same shape, and with the least recently used shape dropped."""
    cases = [case(0, T) for T in range(3, 3 + HipAllToAll.MAX_CACHED_SHAPES)]
    ata = HipAllToAll(cases[0][0], 0, 8, fuse_stub=True)
    for _, rd, _, want in cases + cases:  # both sets of every shape
        assert same(ata.forward(rd.x, rd.indices, rd.weights), want)
        assert same(custom_kernel((cases[0][0], rd, 0, 8)), want)
    built = []
    args, record = HipAllToAll._forward_args, HipAllToAll._record
    monkeypatch.setattr(HipAllToAll, "_forward_args", lambda *a: built.append("block") or args(*a))
    monkeypatch.setattr(HipAllToAll, "_record", lambda *a: built.append("record") or record(*a))
    for turn in range(3):
        for _, rd, _, want in cases if turn else reversed(cases):
            y = ata.forward(rd.x, rd.indices, rd.weights)
            assert same(y, want) and ata.last.num_tokens == y.shape[0]
            first = ata.last.disp_x.data_ptr()
            assert ata.dispatch(rd.x, rd.indices).disp_x.data_ptr() != first  # the other of the two sets
            assert same(custom_kernel((cases[0][0], rd, 0, 8)), want)
    assert not built
    # the shape used longest ago, by a forward or by a dispatch, makes room for a new one
    order = cases[4:] + cases[:4]
    for i, (_, rd, _, _) in enumerate(order):
        ata.dispatch(rd.x, rd.indices) if i % 2 else ata.forward(rd.x, rd.indices, rd.weights)
    _, rd, _, want = case(0, 40)
    assert same(ata.forward(rd.x, rd.indices, rd.weights), want) and built
    kept = {key[0] for key in ata._bufs}
    assert kept == {40} | {c[1].num_tokens for c in order[1:]}
    del built[:]
    for _, rd, _, want in order[1:]:
        assert same(ata.forward(rd.x, rd.indices, rd.weights), want)
    assert not built
    ata.release_buffers()
    _, rd, _, want = cases[0]
    assert same(ata.forward(rd.x, rd.indices, rd.weights), want) and len(ata._bufs) == 1


def test_two_threads_share_a_handle(gpu_device):
    """Two threads call custom_kernel with one configuration, each with token counts of its own in turn, and forward of
    one host object with results of their own: every result is that of its call."""
    import threading

    cfg = case(0, 5)[0]
    cases = {0: [case(0, T) for T in (5, 9, 21)], 1: [case(0, T) for T in (6, 9, 33)]}
    ata = HipAllToAll(cfg, 0, 8, fuse_stub=True)
    wrong = []

    def work(me):
        try:
            kept = []
            for i in range(150):
                _, rd, _, want = cases[me][i % 3]
                kept.append((custom_kernel((cfg, rd, 0, 8)), want))
                out = torch.empty_like(kept[-1][0])
                assert ata.forward(rd.x, rd.indices, rd.weights, out=out) is out
                kept.append((out, want))
            torch.cuda.synchronize()
            wrong.extend(me for y, want in kept if not same(y, want))
        except Exception as e:  # an assertion in a thread is not seen by itself
            wrong.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
