"""The calls that a user of this package has it do, with the inputs they meet in use, for timing.

Four kinds, each through its public entry point:

* ``kernel``   ``custom_kernel(data)``: one rank's tokens through dispatch, expert stand-in and combine, the call
               that the evaluation harness makes;
* ``forward``  ``HipAllToAll.forward``: the same for every rank of a world at once (``rank_start``), or with fp8
               rows; the dispatched buffers of the call belong to its result;
* ``layer``    a real expert layer: ``dispatch`` -> ``expert_gemm`` (hidden -> hidden) -> ``combine``, with 16-bit
               weights, with block-quantised fp8 weights, and with fp8 rows as well;
* ``gemm_rs``  ``HipGemmReduceScatter.forward``: a linear layer whose K is split over the ranks.

The model shapes (experts, top-k, hidden) are those of the benchmark specs in ``kernel_amd/contract.py`` and
``kernel_amd/gemm_rs.py``; token counts run from one decode step to a prefill batch.
"""
import math

import torch

from kernel_amd import gemm_rs
from kernel_amd.all2all import HipAllToAll
from kernel_amd.contract import COMBINE_F32, COMBINE_STRICT, STUB_EXPERT_FRACTION, MoEConfig, RankData
from kernel_amd.submission import custom_kernel

WORLD = 8
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
# (experts, top-k, hidden) of the benchmark specs
SHAPES = ((8, 2, 6144), (64, 6, 2048), (128, 4, 2880), (128, 8, 4096), (256, 8, 7168))
# what the experts of a layer are made of: 16-bit rows and weights; 16-bit rows, fp8 weights; fp8 rows and weights
# with f32 scales; the same with power-of-two scales
FORMATS = ("16bit", "w8", "fp8", "pow2")
MAX_ROW_BYTES = 1.1e9  # of a forward's dispatched rows in 16 bits
MAX_LAYER_FLOPS = 3.3e12
MAX_LAYER_WEIGHT_BYTES = 14e9


def _kernel(name, shape, tokens, dtype):
    return dict(name=name, kind="kernel", experts=shape[0], topk=shape[1], hidden=shape[2], tokens=tokens, dtype=dtype)


def _forward(name, shape, tokens, dtype="bf16", ranks=1, zipf=0.0, fp8="no", combine="strict"):
    return dict(name=name, kind="forward", experts=shape[0], topk=shape[1], hidden=shape[2], tokens=tokens,
                dtype=dtype, ranks=ranks, zipf=zipf, fp8=fp8, combine=combine)


def _layer(name, shape, tokens, form, dtype="bf16", zipf=0.0):
    return dict(name=name, kind="layer", experts=shape[0], topk=shape[1], hidden=shape[2], tokens=tokens, form=form,
                dtype=dtype, zipf=zipf)


def _gemm(name, m, n, k, bias, dtype="bf16"):
    return dict(name=name, kind="gemm_rs", m=m, n=n, k=k, bias=bias, dtype=dtype)


def listed():
    return [
        # the smallest call the harness makes: a handful of tokens, where the launch and the host side are all there is
        _kernel("kernel_e8_t7", (8, 2, 6144), 7, "fp16"),
        # one rank's decode step of a 256-expert model: the headline benchmark
        _kernel("kernel_e256_t256", (256, 8, 7168), 256, "bf16"),
        # a whole world of 8 ranks with unequal token counts and popular experts
        _forward("forward_world_t1003", (64, 6, 2048), 1003, ranks=8, zipf=1.2),
        # a prefill batch through the stand-in: far beyond the caches
        _forward("forward_prefill_t16384", (128, 4, 4096), 16384),
        # decode, 16-bit weights: six rows per expert, every weight is read for them
        _layer("layer_decode_bf16_t96", (128, 8, 4096), 96, "16bit"),
        # decode of a large model with fp8 rows and weights: two rows per expert
        _layer("layer_decode_fp8_t61", (256, 8, 7168), 61, "fp8"),
        # prefill, 16-bit
        _layer("layer_prefill_bf16_t16384", (128, 4, 4096), 16384, "16bit"),
        # a batch of a large model in fp8 with f32 scales: 128 rows per expert
        _layer("layer_batch_fp8_t4096", (256, 8, 7168), 4096, "fp8"),
        # prefill in fp8 with power-of-two scales, ragged segments of some 281 rows
        _layer("layer_prefill_pow2_t9001", (128, 4, 4096), 9001, "pow2"),
        # few rows against a wide weight: reading the weights once
        _gemm("gemm_rs_64x7168x18432", 64, 7168, 18432, False),
        # a mid-size layer whose local K (360) is no multiple of a slab
        _gemm("gemm_rs_2048x2880x2880", 2048, 2880, 2880, True),
        # the largest of the specs (local K 3696)
        _gemm("gemm_rs_8192x8192x29568", 8192, 8192, 29568, False),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("kernel", "kernel", "forward", "forward", "layer", "layer", "layer", "gemm_rs", "gemm_rs"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind == "kernel":
        c = _kernel("", rng.choice(SHAPES), _log_int(rng, 1, 512), dtype)
    elif kind == "forward":
        shape = rng.choice(SHAPES)
        most = min(16384, int(MAX_ROW_BYTES / (2 * shape[1] * shape[2])))
        fp8 = rng.choice(("no", "no", "f32", "pow2")) if shape[2] % 128 == 0 else "no"
        c = _forward("", shape, _log_int(rng, 32, most), dtype, rng.choice((1, WORLD)), rng.choice((0.0, 1.2)), fp8,
                     rng.choice(("strict", "f32")))
    elif kind == "layer":
        form = rng.choice(FORMATS)
        per = 2 if form == "16bit" else 1
        shape = rng.choice([s for s in SHAPES[1:] if (form == "16bit" or s[2] % 128 == 0)
                            and per * s[0] * s[2] * s[2] <= MAX_LAYER_WEIGHT_BYTES])
        most = min(16384, int(MAX_LAYER_FLOPS / (2 * shape[1] * shape[2] * shape[2])))
        c = _layer("", shape, _log_int(rng, 8, most), form, dtype, rng.choice((0.0, 0.0, 1.2)))
    else:
        c = _gemm("", 8 * _log_int(rng, 4, 1024), 64 * _log_int(rng, 32, 128), 64 * _log_int(rng, 32, 462),
                  rng.random() < 0.5, dtype)
    del c["name"]
    return c


def _routing(c, dev, gen):
    """Expert ids without replacement: uniform, or popularity ~ rank^-zipf (Gumbel top-k of the log weights)."""
    T, E, K = c["tokens"], c["experts"], c["topk"]
    score = -torch.log(-torch.log(torch.rand(T, E, device=dev, generator=gen).clamp_(1e-9, 1 - 1e-7)))
    if c.get("zipf"):
        score -= c["zipf"] * torch.log(torch.arange(1, E + 1, device=dev, dtype=torch.float32))
    return score.topk(K, dim=1).indices.to(torch.int32).contiguous()


def _expert_weights(c, dev, gen):
    """(weights[E, N, H], w_scale or None), N == H, of the size a trained layer has: N(0, 1/H)."""
    E, H = c["experts"], c["hidden"]
    if c["form"] == "16bit":
        w = torch.empty(E, H, H, dtype=DTYPES[c["dtype"]], device=dev)
        for e in range(E):
            w[e].normal_(0.0, H ** -0.5, generator=gen)
        return w, None
    w = torch.empty(E, H, H, dtype=torch.float8_e4m3fn, device=dev)
    block = torch.empty(H, H, dtype=torch.bfloat16, device=dev)
    for e in range(E):
        # a block of 128 x 128 has its largest value, some four standard deviations, near the format's 448
        w[e] = block.normal_(0.0, 448 / 4.5, generator=gen).clamp_(-448, 448).to(torch.float8_e4m3fn)
    shape = (E, H // 128, H // 128)
    base = H ** -0.5 * 4.5 / 448
    if c["form"] == "pow2":
        scale = torch.exp2(torch.randint(-1, 2, shape, device=dev, generator=gen).float() + round(math.log2(base)))
    else:
        scale = base * (0.75 + 0.5 * torch.rand(shape, device=dev, generator=gen))
    return w, scale.contiguous()


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    c, dt = dict(case), DTYPES[case["dtype"]]
    if c["kind"] == "gemm_rs":
        kl = c["k"] // WORLD
        x = torch.empty(WORLD, c["m"], kl, dtype=dt, device=dev).uniform_(-0.01, 0.01, generator=gen)
        w = torch.empty(WORLD, c["n"], kl, dtype=dt, device=dev).uniform_(-0.01, 0.01, generator=gen)
        bias = torch.empty(c["n"], dtype=dt, device=dev).uniform_(-0.01, 0.01, generator=gen) if c["bias"] else None
        return dict(c, handle=gemm_rs.HipGemmReduceScatter(WORLD), x=x, w=w, bias_t=bias)
    T, E, K, H = c["tokens"], c["experts"], c["topk"], c["hidden"]
    x = torch.randn(T, H, device=dev, generator=gen)
    rows = torch.randperm(T, device=dev, generator=gen)[: T // 100]
    x[rows] *= 100.0  # the outlier tokens of a long batch
    x = x.to(dt)
    idx = _routing(c, dev, gen)
    cfg = MoEConfig(E, K, H, max_num_tokens=T + 1, in_dtype=dt, out_dtype=dt)
    if c["kind"] == "kernel":
        w = torch.rand(T, K, device=dev, generator=gen)
        return dict(c, data=(cfg, RankData(T, idx, w, x), seed % WORLD, WORLD))
    w = torch.softmax(torch.randn(T, K, device=dev, generator=gen), dim=-1)
    if c["kind"] == "forward":
        ata = HipAllToAll(cfg, 0, WORLD, stub_kind=STUB_EXPERT_FRACTION, fuse_stub=True,
                          combine_mode=COMBINE_STRICT if c["combine"] == "strict" else COMBINE_F32,
                          fp8_dispatch={"no": False, "f32": True, "pow2": "pow2"}[c["fp8"]])
        starts = None
        if c["ranks"] > 1:
            cuts = torch.randint(0, T + 1, (c["ranks"] - 1,), device=dev, generator=gen).sort().values
            starts = torch.cat([cuts.new_zeros(1), cuts, cuts.new_full((1,), T)]).to(torch.int32)
        return dict(c, ata=ata, x=x, idx=idx, w=w, starts=starts)
    ata = HipAllToAll(cfg, 0, WORLD, fp8_dispatch={"fp8": True, "pow2": "pow2"}.get(c["form"], False))
    weights, w_scale = _expert_weights(c, dev, gen)
    return dict(c, ata=ata, x=x, idx=idx, w=w, weights=weights, w_scale=w_scale)


def _buffers(d):
    """The dispatched buffers of a call: segment table, permutation, meta rows, rows, scales."""
    return dict(counts=d.counts, offsets=d.offsets, slot=d.slot_of_entry, src=d.src_of_slot, meta=d.meta, rows=d.disp_x,
                scale=d.disp_scale)


def run(s):
    if s["kind"] == "kernel":
        return custom_kernel(s["data"])
    if s["kind"] == "gemm_rs":
        return s["handle"].forward(s["x"], s["w"], s["bias_t"])
    ata = s["ata"]
    if s["kind"] == "forward":
        y = ata.forward(s["x"], s["idx"], s["w"], s["starts"])
        return dict(_buffers(ata.last), y=y)
    d = ata.dispatch(s["x"], s["idx"])
    ey = ata.expert_gemm(d, s["weights"], w_scale=s["w_scale"], scales_pow2=s["form"] == "pow2")
    return dict(_buffers(d), expert_y=ey, y=ata.combine(None, s["w"], d, ey))


def work(case):
    """Bytes: inputs once, results once; the dispatched rows are a result (each expert's segment), the weights of
    the experts that no token chose are not read."""
    c = case
    if c["kind"] == "gemm_rs":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 2.0 * (m * k + n * k + m * n), "flops": 2.0 * m * n * k}
    T, E, K, H = c["tokens"], c["experts"], c["topk"], c["hidden"]
    R = T * K
    q = c.get("fp8", "no") != "no" or c.get("form") in ("fp8", "pow2")
    row = H + 4 * H // 128 if q else 2 * H
    # x, y; ids and weights; dispatched rows; permutation and meta rows; segment table
    nbytes = 4.0 * T * H + 8.0 * R + float(R) * row + 28.0 * R + 8.0 * E
    if c["kind"] != "layer":
        return {"bytes": nbytes, "flops": 3.0 * R * H}
    chosen = E * (1.0 - (1.0 - K / E) ** T)
    per = 2.0 if c["form"] == "16bit" else 1.0 + 4.0 / (128 * 128)
    nbytes += chosen * per * H * H + 2.0 * R * H
    return {"bytes": nbytes, "flops": 2.0 * R * H * H + 2.0 * R * H}


def tolerance(case):
    # the strict combine is defined bit for bit; the index arrays and the quantised rows are whole values anywhere
    if case["kind"] == "kernel" or case.get("combine") == "strict":
        return "exact"
    # one rounding of the element type per value, another order of the f32 sums before it
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3}
