"""Batches of odd and even numbers of limbs whose descriptors are uploaded by the kernel (more than 16 KB): the
descriptors at the end of the upload, of 8 bytes modulo 16, arrive as the others do."""
import pytest

from gpu_cases import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [90, 91, 92, 93])
def test_batches_of_odd_and_even_limb_totals(count):
    ctx, _ = make(("upload_tail", 12, [50] * 6, [60] * 2, 3))
    key = ctx.ksk_uniform(5, seed=3)
    src = [ctx.uniform(level, seed=20 + level) for level in range(6)]
    want = [[p.digest() for p in ctx.key_switch(d, key)] for d in src]
    levels = [(5 * i + count) % 6 for i in range(count)]
    for _ in range(3):  # direct, captured, replayed
        got = ctx.key_switch_batch([src[x] for x in levels], key)
        for x, (kb, ka) in zip(levels, got):
            assert [kb.digest(), ka.digest()] == want[x], x
