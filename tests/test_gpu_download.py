"""Large downloads go through pinned chunks (lfgpu_core.hip): what arrives is
what was uploaded, bit for bit."""
import threading

import numpy as np
import pytest

from lehrfempp_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with capi.Context(0) as c:
        yield c


# the last plain size (4 MiB less a value), one and two chunks of 2 MiB more or
# less a value, every chunk of the ring and one more, and twice around it
@pytest.mark.parametrize("n", [524287, 524288, 524289, 786431, 786433, 2097152, 2097153, 4456449])
def test_vector_download(ctx, n):
    want = np.random.default_rng(n).standard_normal(n)
    v = capi.Vec(ctx, want)
    for _ in range(2):
        assert np.array_equal(v.numpy(), want)
    v.close()


def test_matrix_download(ctx):
    n = 400000
    i = np.arange(n)
    v = np.random.default_rng(0).standard_normal(3 * n - 2)
    r, c = np.concatenate([i, i[:-1], i[1:]]), np.concatenate([i, i[1:], i[:-1]])
    A = capi.coo_to_csr(ctx, r, c, v, n, n)
    rp, col, val = A.download()
    o = np.lexsort((c, r))
    assert np.array_equal(rp, np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]))
    assert np.array_equal(col, c[o]) and np.array_equal(val, v[o])
    A.close()


def test_downloads_from_two_threads(ctx):
    want = [np.random.default_rng(k).standard_normal(1500000 + k) for k in range(2)]
    vecs = [capi.Vec(ctx, w) for w in want]
    bad = []

    def work(k):
        for _ in range(5):
            if not np.array_equal(vecs[k].numpy(), want[k]):
                bad.append(k)

    team = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad
    for v in vecs:
        v.close()
