"""Where the tile loops of gemm_rs read: on the CPU, from the kernels' own sources.

The loops are cut out of ``kernel_amd/csrc``, compiled for the host with stand-ins for the matrix and buffer instructions
(``tile_loops.py``), and run thread by thread.  Every request inside a buffer has to lie in a row of an operand, and all rows have
to be asked for.  No GPU, and nothing is read from the addresses."""
import random

import pytest

import tile_loops


def launch(form, m, n, kl, W, groups, pitch, cols, at=(0, 0), gap=(0, 0)):
    return (form, m, n, kl, W, groups, pitch, cols, *at, *gap)


def launches(ms, ns, kls, rng):
    """Each form in each of its tile heights on operands of these sizes, at any place within a line, with shards any gap apart."""
    for m in ms:
        for n in ns:
            for kl in kls:
                for W in (1, 2, 8):
                    at, gap = (rng.randrange(8), rng.randrange(8)), (rng.choice((0, 0, 3, 5, 17)), rng.choice((0, 0, 1, 6)))
                    for form in ("wl", "wr"):
                        yield launch(form, m, n, kl, W, 1, rng.choice((256, 192, 128)), 256, at, gap)
                    for groups in {1, W if n % 4 == 0 else 1}:  # (partial products are written four columns at a time)
                        yield launch(rng.choice(("nl", "nr")), m, n, kl, W, groups, rng.choice((256, 192, 128)), 128, at, gap)
                        if m <= 64:
                            yield launch(rng.choice(("rl", "rr")), m, n, kl, W, groups, 64, rng.choice((64, 128)), at, gap)
                    if W > 1 and n % 4 == 0:
                        yield launch(rng.choice(("sl", "sr")), m, n, kl, W, W, rng.choice((256, 208, 16)), rng.choice((256, 176, 64)), at, gap)


def check(cases):
    for case, got in zip(cases, tile_loops.run(cases)):
        requests, outside, missed = map(int, got)
        assert outside == 0 and missed == 0 and requests > 0, (case, requests, outside, missed)


KLS = (64, 72, 80, 96, 104, 128, 136, 184, 192, 200, 264, 312, 360, 456, 712, 720, 776)


@pytest.mark.parametrize("m,n", [(1, 1), (1, 300), (65, 1), (1, 40), (130, 2), (2, 130)])
def test_operands_of_one_row_or_two(m, n):
    """Shards one row apart begin less than a line behind the last one's end: what takes a request there is a step backwards, also
    for the rows that do not exist."""
    check(list(launches([m], [n], KLS, random.Random(m + n))))


@pytest.mark.parametrize("seed", range(4))
def test_any_operands(seed):
    rng = random.Random(seed)
    size = lambda most: int(2 ** rng.uniform(0, most))
    cases = []
    for _ in range(12):
        cases += launches([size(9.2)], [size(9.2)], [8 * rng.randrange(8, 100)], rng)
    check(cases)


def check_calls(cases):
    """(option, m, n, kl, W, at, gap) through gemm_rs_forward, with room for any partial products."""
    lines = [("call", 1, option, m, n, kl, W, *at, *gap, 4 * W * m * n, 0) for option, m, n, kl, W, at, gap in cases]
    for case, got in zip(cases, tile_loops.run(lines)):
        requests, outside, missed = map(int, got[-5:-2])
        assert got[0] == "0" and outside == 0 and missed == 0 and requests > 0, (case, got)


@pytest.mark.parametrize("m,n,kl,W", [(128, 1, 360, 8), (65, 1, 72, 2), (520, 1, 360, 8), (520, 1, 776, 2), (1, 32776, 720, 8), (1, 33000, 712, 1)])
def test_operands_of_one_row_as_the_library_multiplies_them(m, n, kl, W):
    check_calls([(0, m, n, kl, W, (0, 0), (0, 0))])


@pytest.mark.parametrize("seed", range(3))
def test_calls_as_the_library_multiplies_them(seed):
    rng, cases = random.Random(seed), []
    while len(cases) < 24:
        W, m, n, kl = rng.choice((1, 2, 3, 8)), int(2 ** rng.uniform(0, 11)), 4 * int(2 ** rng.uniform(0, 9)), 8 * rng.randrange(8, 70)
        if W * (m + n) * kl <= 4 << 20:
            cases.append((rng.choice((0, 0, 256, 129, 130, 131, 132, 133)), m, n, kl, W, (rng.randrange(8), rng.randrange(8)), (rng.choice((0, 3)), rng.choice((0, 6)))))
    check_calls(cases)


FAR = 1 << 27  # 16-byte vectors: 2 GiB


@pytest.mark.parametrize("gap", [(FAR, FAR), (FAR, 0), (0, FAR), (FAR - 40000, 5), (FAR // 2, FAR - 70000)])
@pytest.mark.parametrize("form,m,n,kl", [(256, 300, 264, 712), (129, 300, 264, 776), (131, 400, 264, 360), (132, 130, 264, 72), (130, 300, 132, 456),
                                         (133, 300, 264, 712), (0, 37, 16, 712)])
def test_shards_far_apart(form, m, n, kl, gap):
    """Further than a 32-bit offset reaches, or just not."""
    check_calls([(form, m, n, kl, W, (3, 5), gap) for W in (2, 7)])
