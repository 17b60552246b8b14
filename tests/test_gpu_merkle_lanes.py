"""Merkle forests at the sizes where the number of lanes per leaf and per node
changes (16 lanes, a quad, one lane), through the ABI (row-major leaves) and
the fused commit (column-major LDE), bit-exact against the oracle."""
import numpy as np
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


# leaf counts on both sides of 2^13 and 2^16; sizes of one chunk, a whole
# second chunk, and last chunks of 1, 3, 4 and 7 elements
@pytest.mark.parametrize("n_leaves,leaf_size,cap_height", [
    (2, 5, 0), (4, 9, 1), (1 << 13, 8, 4), (1 << 13, 23, 0), (1 << 14, 17, 3), (1 << 14, 11, 13),
    (1 << 16, 12, 2), (1 << 17, 16, 5),
])
def test_row_major_forest(Z, n_leaves, leaf_size, cap_height):
    from gpu_util import dev, empty, host
    leaves = O.random(n_leaves * leaf_size, 900 + n_leaves + leaf_size)
    nd, nc = 2 * (n_leaves - (1 << cap_height)), 1 << cap_height
    dl, dd, dc = dev(leaves), empty(4 * nd), empty(4 * nc)
    Z.fill_digests_buf_linear_gpu_with_gpu_ptr(dd, dc, dl, nd, nc, n_leaves, leaf_size, cap_height)
    odg, ocp = O.merkle(leaves, n_leaves, leaf_size, cap_height)
    assert (host(dc) == ocp).all()
    assert (host(dd, 4 * nd) == odg).all()


@pytest.mark.parametrize("lg_n,r,C,h,rows", [
    (4, 1, 9, 2, True), (10, 3, 20, 4, False), (10, 3, 13, 4, True), (11, 3, 17, 4, True), (13, 3, 9, 2, True),
])
def test_commit_forest(Z, lg_n, r, C, h, rows):
    from gpu_util import dev, empty, host
    N = 1 << (lg_n + r)
    coeffs = O.random(C << lg_n, 950 + lg_n + C)
    nd = 2 * (N - (1 << h))
    lde, lv, dg, cp = empty(C * N), (empty(C * N) if rows else None), empty(4 * nd), empty(4 << h)
    Z.commit(0, dev(coeffs), lde, lv, dg, cp, lg_n, r, C, h)
    leaves = O.transpose_rev(O.lde(coeffs, lg_n, r, C), lg_n + r, C)
    odg, ocp = O.merkle(leaves, N, C, h)
    if rows:
        assert (host(lv) == leaves).all()
    assert (host(cp) == ocp).all() and (host(dg) == odg).all()


@pytest.mark.parametrize("n_leaves,leaf_size", [(512, 12), (1 << 14, 16), (1 << 17, 21)])
def test_rare_case_leaves(Z, n_leaves, leaf_size):
    """Leaves that take the exact recompute path in the 16-lane, quad and
    one-lane kernels, also in a chunk that is not the last."""
    from gpu_util import dev, empty, host
    from rare_inputs import leaves_with_rare_cases
    leaves = leaves_with_rare_cases(O.random(n_leaves * leaf_size, 77 + n_leaves), n_leaves, leaf_size)
    nd = 2 * (n_leaves - 4)
    dl, dd, dc = dev(leaves), empty(4 * nd), empty(16)
    Z.fill_digests_buf_linear_gpu_with_gpu_ptr(dd, dc, dl, nd, 4, n_leaves, leaf_size, 2)
    odg, ocp = O.merkle(leaves, n_leaves, leaf_size, 2)
    assert (host(dc) == ocp).all() and (host(dd, 4 * nd) == odg).all()


@pytest.mark.parametrize("leaf_size", [3, 4, 16, 17, 18, 33, 34, 35])
def test_keccak_leaf_sizes(Z, leaf_size):
    """Keccak leaves whose last block holds no, one, and all but one of the
    17 words beside the padding; two-leaf subtrees and one deeper forest."""
    from gpu_util import dev, empty, host
    for n, h in ((64, 5), (256, 2)):
        leaves = O.random(n * leaf_size, 40 + leaf_size)
        nd = 2 * (n - (1 << h))
        dl, dd, dc = dev(leaves), empty(4 * nd), empty(4 << h)
        Z.fill_digests_buf_linear_gpu_with_gpu_ptr(dd, dc, dl, nd, 1 << h, n, leaf_size, h, hash_type=1)
        odg, ocp = O.merkle(leaves, n, leaf_size, h, hash_type=1)
        assert (host(dc) == ocp).all() and (host(dd, 4 * nd) == odg).all()
