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
                        yield launch("n", m, n, kl, W, groups, rng.choice((256, 192, 128)), 128, at, gap)
                        if m <= 64:
                            yield launch(rng.choice(("rl", "rr")), m, n, kl, W, groups, 64, rng.choice((64, 128)), at, gap)
                    if W > 1 and n % 4 == 0:
                        yield launch("s", m, n, kl, W, W, rng.choice((256, 208, 16)), rng.choice((256, 176, 64)), at, gap)


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


@pytest.mark.parametrize("m,n,kl,W,form,pitch,cols", [
    (128, 1, 360, 8, "n", 128, 128), (65, 1, 72, 2, "n", 128, 128), (520, 1, 360, 8, "n", 256, 128),
    (1, 32776, 720, 8, "wl", 256, 256), (1, 33000, 712, 1, "wl", 256, 256),
])
def test_operands_of_one_row_as_the_library_multiplies_them(m, n, kl, W, form, pitch, cols):
    check([launch(form, m, n, kl, W, 1, pitch, cols)])
