"""Batches whose launches lie exactly at, and one limb beyond, the limits at which the narrow and the 16-word
passes, the fused conversions and the inner product inside the row passes change over: every switch of a batch gives
the words of the same switch alone, which are the oracle's. The limits are in tiles of 4096 words."""
import pytest

import ckh
import oracle as O
from gpu_cases import make

pytestmark = pytest.mark.gpu

ROWS, COLS8, ALONE, IP, CONV = 4096, 320, 128, 1024, 8192
# Limbs per switch of one limb in each kind of launch (alpha 1, two special primes): the inverse transform of the
# input, the forward transforms and conversion targets, the inverse transforms of both parts' special limbs.
RATES = {"input": 1, "targets": 2, "special": 4}


def tiles(log_n, limbs):
    return limbs << (log_n - 12)


def batch_counts(log_n, limit, rate):
    """The switches of the batch at the limit and of the one beyond it."""
    at = (limit >> (log_n - 12)) // rate
    assert tiles(log_n, rate * at) <= limit < tiles(log_n, rate * (at + 1))
    return at, at + 1


def check_batches(ctx, ref, level, counts):
    key = ctx.ksk_uniform(len(ref.q) - 1, seed=31)
    polys = [ctx.uniform(level, seed=400 + i) for i in range(3)]
    want = [[p.digest() for p in ctx.key_switch(d, key)] for d in polys]
    kb, ka = ctx.key_switch(polys[0], key)
    wb, wa = ref.key_switch(polys[0].download().ravel(), level, ref.uniform_key(len(ref.q) - 1, 31), len(ref.q) - 1)
    assert (kb.download() == wb).all() and (ka.download() == wa).all()
    for count in sorted(counts):
        got = ctx.key_switch_batch([polys[i % 3] for i in range(count)], key)
        for i in sorted({*range(0, count, 7), count - 2, count - 1}):
            assert [p.digest() for p in got[i]] == want[i % 3], (count, i)
        del got


@pytest.mark.parametrize("q_bits", [50, 60])
@pytest.mark.parametrize("log_n, limit", [(n, ROWS) for n in range(12, 17)] + [(n, COLS8) for n in (15, 16)] +
                         [(n, IP) for n in range(12, 17)])
def test_batches_at_the_limits(log_n, limit, q_bits):
    ctx, ref = make(("limits", log_n, [q_bits] * 2, [60] * 2, 2))
    rates = {"targets": RATES["targets"]} if limit == IP else RATES
    check_batches(ctx, ref, 0, {c for r in rates.values() for c in batch_counts(log_n, limit, r)})


@pytest.mark.parametrize("log_n", [12, 14, 16])
def test_fused_conversions_at_their_limit(log_n):
    """Six sources: fused up to 8192 tiles of targets (six of ModUp, eight of mod_down at four limbs)."""
    ctx, ref = make(("limits6", log_n, [50] * 6, [60] * 6, 1))
    check_batches(ctx, ref, 3, {c for r in (6, 8) for c in batch_counts(log_n, CONV, r)})


@pytest.mark.parametrize("log_n", [14, 15, 16])
def test_plain_transforms_at_their_limit(log_n):
    at = ALONE >> (log_n - 12)
    assert tiles(log_n, at) == ALONE
    q = O.ntt_primes(50, 1 << log_n, at + 1)
    ctx = ckh.Context(log_n, q, O.ntt_primes(60, 1 << log_n, 1), at + 1)
    for limbs in (at, at + 1):
        a = O.uniform_poly(q[:limbs], 1 << log_n, limbs)
        f = ctx.upload(a, limbs - 1, ntt=False).ntt()
        assert (f.download() == O.ntt_forward(1 << log_n, q[:limbs], a.ravel()).reshape(limbs, -1)).all()
        assert (f.intt().download() == a).all()
