"""Uploads on each side of the sizes at which the way changes (copy command, kernel, DMA in pieces): the words
that come back are those sent, several uploads in a row without a wait between them."""
import numpy as np
import pytest

from gpu_cases import host_uniform, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n, limbs", [(10, 1), (10, 2), (10, 3), (11, 5), (14, 7), (14, 8), (14, 9), (16, 24)])
def test_uploaded_words_come_back(log_n, limbs):
    ctx, ref = make(("upload", log_n, [50] * 24, [60] * 6, 4))
    sent = [host_uniform(ref, limbs - 1, 60 + i) for i in range(4)]
    polys = [ctx.upload(a, limbs - 1) for a in sent]
    for a, p in zip(sent, polys):
        assert (p.download() == np.asarray(a).reshape(limbs, -1)).all()
