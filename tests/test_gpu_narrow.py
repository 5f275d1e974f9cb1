"""The narrow passes on the device: one switch (narrow passes, inner product inside the row passes) and a
batch beyond each limit (16-word passes, inner product of its own) give the oracle's words, at every ring size."""
import pytest

from gpu_cases import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n, count", [(12, 900), (13, 450), (14, 230), (15, 120), (16, 60)])
def test_narrow_and_wide_launches_equal_the_oracle(log_n, count):
    ctx, ref = make(("narrow", log_n, [60, 50, 40], [60, 60], 3))
    key = ctx.ksk_uniform(2, seed=31)
    polys = [ctx.uniform(i % 3, seed=400 + i) for i in range(6)]
    one = [tuple(k.download() for k in ctx.key_switch(p, key)) for p in polys]
    wb, wa = ref.key_switch(polys[2].download().ravel(), 2, ref.uniform_key(2, 31), 2)
    assert (one[2][0] == wb).all() and (one[2][1] == wa).all()
    got = ctx.key_switch_batch([polys[2 - i % 2] for i in range(count)], key)
    for i in {0, 1, count - 2, count - 1}:
        kb, ka = got[i]
        want = one[2 - i % 2]
        assert (kb.download() == want[0]).all() and (ka.download() == want[1]).all(), i
    back = polys[2].intt().ntt().download()
    assert (back == polys[2].download()).all()
