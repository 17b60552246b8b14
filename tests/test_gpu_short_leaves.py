"""Leaves of at most four elements, which are copied instead of hashed: every
size, all leaves caps or levels above them, partial last workgroups, through
the ABI, the fused commit with and without leaf rows, and a batch."""
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Z():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import zeknox_amd
    zeknox_amd.init_cuda_rs()
    return zeknox_amd


@pytest.mark.parametrize("leaf_size", [1, 2, 3, 4])
@pytest.mark.parametrize("lg,h", [(0, 0), (1, 0), (5, 5), (5, 1), (9, 9), (11, 3), (17, 16)])
def test_row_major(Z, leaf_size, lg, h):
    import torch
    from gpu_util import dev, empty, host
    n, nd = 1 << lg, 2 * ((1 << lg) - (1 << h))
    leaves = O.random(n * leaf_size, 1400 + 8 * lg + leaf_size)
    dl, dd, dc = dev(leaves), empty(4 * nd), empty(4 << h)
    dd.fill_(-1)
    dc.fill_(-1)
    torch.cuda.synchronize()
    Z.fill_digests_buf_linear_gpu_with_gpu_ptr(dd, dc, dl, nd, 1 << h, n, leaf_size, h)
    odg, ocp = O.merkle(leaves, n, leaf_size, h)
    assert (host(dc) == ocp).all() and (host(dd, 4 * nd) == odg).all()


@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("lg_n,r,C,h", [(4, 1, 1, 5), (4, 1, 3, 2), (10, 3, 4, 13), (9, 2, 2, 0), (13, 3, 3, 4)])
def test_commit(Z, lg_n, r, C, h, rows):
    from gpu_util import dev, empty, host
    N = 1 << (lg_n + r)
    coeffs = O.random(C << lg_n, 1500 + lg_n + C)
    nd = 2 * (N - (1 << h))
    lde, lv, dg, cp = empty(C * N), (empty(C * N) if rows else None), empty(4 * nd), empty(4 << h)
    Z.commit(0, dev(coeffs), lde, lv, dg, cp, lg_n, r, C, h)
    leaves = O.transpose_rev(O.lde(coeffs, lg_n, r, C), lg_n + r, C)
    odg, ocp = O.merkle(leaves, N, C, h)
    if rows:
        assert (host(lv) == leaves).all()
    assert (host(cp) == ocp).all() and (host(dg, 4 * nd) == odg).all()


def test_batch_beside_hashed_leaves(Z):
    """Jobs of copied and of hashed leaves in one launch."""
    import torch
    from gpu_util import dev, empty, host
    jobs, bufs = [], []
    for lg_n, r, C, h in ((6, 1, 4, 3), (8, 2, 9, 2), (5, 3, 1, 8), (9, 1, 3, 0), (7, 1, 5, 4)):
        N = 1 << (lg_n + r)
        c = O.random(C << lg_n, 1600 + lg_n + C)
        b = dict(coeffs=dev(c), lde=empty(C * N), leaves=empty(C * N), digests=empty(8 * (N - (1 << h))),
                 cap=empty(4 << h))
        jobs.append(dict(lg_n=lg_n, rate_bits=r, ncols=C, cap_height=h, **{k: v.data_ptr() for k, v in b.items()}))
        bufs.append((c, b, lg_n, r, C, h))
    torch.cuda.synchronize()
    Z.batch_commit(0, jobs)
    torch.cuda.synchronize()
    for c, b, lg_n, r, C, h in bufs:
        N = 1 << (lg_n + r)
        leaves = O.transpose_rev(O.lde(c, lg_n, r, C), lg_n + r, C)
        odg, ocp = O.merkle(leaves, N, C, h)
        nd = 2 * (N - (1 << h))
        assert (host(b["leaves"]) == leaves).all() and (host(b["cap"]) == ocp).all()
        assert (host(b["digests"], 4 * nd) == odg).all()
