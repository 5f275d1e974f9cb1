"""The no-allocation batched switch close to its fixed workspace: batches whose scratch leaves little room for
the descriptors still run (with the programs that need the fewest descriptor bytes), word for word."""
import random

import pytest

from gpu_cases import make

pytestmark = pytest.mark.gpu

WORKSPACE = 256 << 20  # CKH_STATIC_SCRATCH_BYTES
SHAPES = [((50,) * 24, (60,) * 6, 4), ((50,) * 6, (60,) * 2, 3), ((60, 40, 40, 40), (60,), 4)]


def full_batch(shape, room, log_n=12):
    """Limb counts whose scratch leaves exactly `room` bytes of the workspace."""
    qb, pb, dnum = shape
    top, k, alpha = len(qb), len(pb), len(qb) // dnum

    def scratch(limbs):
        return (limbs + -(-limbs // alpha) * (limbs + k) + 2 * (limbs + k) + 2 * k + 2 * limbs) << (log_n + 3)

    rng = random.Random(3)
    while True:
        limbs, left = [], WORKSPACE
        while left >= scratch(top):
            limbs.append(rng.randint(1, top))
            left -= scratch(limbs[-1])
        for x in range(top, 0, -1):
            while left - scratch(x) >= room:
                limbs.append(x)
                left -= scratch(x)
        if left == room:
            return limbs


@pytest.mark.parametrize("shape, room", list(zip(SHAPES, (327680, 327680, 425984))))
def test_batches_that_nearly_fill_the_workspace_run(shape, room):
    qb, pb, dnum = shape
    ctx, _ = make(("limit", 12, list(qb), list(pb), dnum))
    key = ctx.ksk_uniform(len(qb) - 1, seed=5)
    src = [ctx.uniform(i, seed=9 + i) for i in range(len(qb))]
    limbs = full_batch(shape, room)
    outs = [(ctx.uniform(x - 1, seed=1), ctx.uniform(x - 1, seed=2)) for x in limbs]
    ctx.key_switch_batch_static([src[x - 1] for x in limbs], key, outs)
    want = {x: [p.digest() for p in ctx.key_switch(src[x - 1], key)] for x in set(limbs)}
    for x, (kb, ka) in zip(limbs, outs):
        assert [kb.digest(), ka.digest()] == want[x], x
