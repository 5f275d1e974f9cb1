"""Products with encrypted diagonals whose blocks are taken in several groups, in one, and alone: the words of the
same product put together call by call."""
import pytest

import ckh
from gpu_cases import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("baby, giant, offset", [(2, 16, 0), (1, 8, -1), (2, 4, -3), (4, 1, 0), (4, 1, -1), (8, 32, 0)])
def test_grouped_blocks_equal_single_calls(baby, giant, offset):
    ctx, _ = make(("enc_groups", 12, [50] * 6, [60] * 2, 3))
    steps = sorted({k for k in range(1, baby)} | {offset + baby * k for k in range(giant)} - {0})
    keys = [ctx.ksk_uniform(5, seed=70 + i, galois=ckh.galois_elt(12, s)) for i, s in enumerate(steps)]
    ev = ckh.Evaluator(ctx, ctx.ksk_uniform(5, seed=9), keys)

    def ct(seed):
        return ctx.ct_from_polys([ctx.uniform(4, seed=seed, stream0=100 * c) for c in range(2)], 2.0 ** 40)

    x = ct(1)
    entries = [ct(100 + i) if (i * 7) % 5 else None for i in range(baby * giant)]
    xs = ev.hoisted_rotate(x, list(range(baby)))
    total = None
    for k1 in range(giant):
        block = None
        for k2 in range(baby):
            e = entries[k1 * baby + k2]
            if e is not None:
                p = ev.mul_no_relin(e, xs[k2])
                block = p if block is None else ev.add(block, p)
        if block is None:
            continue
        block = ev.rotate(ev.relinearize(block), offset + baby * k1)
        total = block if total is None else ev.add(total, block)
    for _ in range(3):
        assert (ev.matvec_enc(x, entries, baby, giant, 1, offset).download() == total.download()).all()
