"""The 9-bit and 8-bit forms of the 16-element NTT kernel on the GPU in the
roles that the shipped plans reach for few sizes only: the exact path of the
8-bit first pass, and 9-bit passes after the first."""
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


@pytest.fixture
def plan(Z):
    """Sets the plan of a size; the one that was loaded comes back at the end."""
    saved = {}

    def set_plan(lg, *p):
        saved.setdefault(lg, Z.ntt_tune_get(lg))
        Z.ntt_tune_set(lg, *p)
    yield set_plan
    for lg, p in saved.items():
        Z.ntt_tune_set(lg, *p) if p else Z.ntt_tune_set(lg)


# 16 columns of 2^18 points as 8 + 10 bits: 512 workgroups, the fewest with
# which the first pass takes the 8-bit form
@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("direction,rate", [(0, 0), (1, 0), (0, 3)])
def test_first_8bit_pass_equals_oracle(Z, plan, monkeypatch, direction, rate, force):
    from gpu_util import dev, empty, host
    lg, C = 18, 16
    plan(lg, (8, 10), (-1, -1), (1, 1))
    if force:
        monkeypatch.setenv("ZK_NTT_FORCE_EXACT", "1")
    x = O.random(C << (lg - rate), 1200 + 2 * direction + rate)
    print("8-bit form", direction, rate, force, flush=True)
    cfg = Z.NTTConfig(batches=C, extension_rate_bits=rate, with_coset=rate > 0, are_inputs_on_device=True,
                      are_outputs_on_device=True)
    if rate:
        out = empty(C << lg)
        Z.lde_batch(0, out, dev(x), lg - rate, cfg)
        assert (host(out) == O.lde(x, lg - rate, rate, C)).all()
    else:
        out = dev(x)
        (Z.intt_batch if direction else Z.ntt_batch)(0, out, lg, cfg)
        assert (host(out) == O.ntt(x, lg, C, inverse=bool(direction))).all()


@pytest.mark.parametrize("lg,C,bits", [(18, 17, (9, 9)), (19, 5, (10, 9)), (17, 3, (8, 9)), (22, 2, (4, 9, 9))])
@pytest.mark.parametrize("force", [False, True])
def test_later_9bit_pass_equals_general_pass(Z, plan, monkeypatch, lg, C, bits, force):
    """The same plan with the general kernel (itself pinned to the oracle by
    test_gpu_ntt.py), forward and inverse; the round trip gives the input."""
    import torch
    from gpu_util import empty
    x = empty(C << lg)
    Z.fill_random(0, x, C << lg, 1300 + lg)
    cfg = Z.NTTConfig(batches=C, are_inputs_on_device=True, are_outputs_on_device=True)
    auto = (-1,) * len(bits)
    out = {}
    if force:
        monkeypatch.setenv("ZK_NTT_FORCE_EXACT", "1")
    print("9-bit form", lg, C, bits, force, flush=True)
    for k in (0, 1):
        plan(lg, bits, auto, tuple(k if b == 9 else 1 for b in bits))
        y = x.clone()
        torch.cuda.synchronize()
        Z.ntt_batch(0, y, lg, cfg)
        z = x.clone()
        torch.cuda.synchronize()
        Z.intt_batch(0, z, lg, cfg)
        torch.cuda.synchronize()
        out[k] = (y.clone(), z)
        torch.cuda.synchronize()
        Z.intt_batch(0, y, lg, cfg)
        torch.cuda.synchronize()
        assert torch.equal(y, x), (lg, bits, k)
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), (lg, bits)
