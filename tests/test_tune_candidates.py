"""The plans the NTT autotuner offers: for every pass that the 16-element
kernel may run, that kernel and the general one."""
import pytest

from zeknox_amd import tune


def switchable(bits):
    """Passes whose 16-element kernel flag means something."""
    return [p for p, b in enumerate(bits) if b in (9, 10) or (b == 8 and p == 0)]


@pytest.mark.parametrize("lg,bits", [(18, (9, 9)), (18, (8, 10)), (17, (9, 8)), (19, (10, 9)), (21, (8, 5, 8)),
                                     (20, (10, 10)), (24, (8, 8, 8))])
def test_both_kernels_are_offered(lg, bits):
    flags = {k for b, _, k in tune.candidates(lg) if b == bits}
    assert (1,) * len(bits) in flags
    for p in switchable(bits):
        assert any(k[p] == 0 for k in flags), (bits, p)


@pytest.mark.parametrize("lg", [5, 8, 9, 10, 13, 16, 18, 21])
def test_candidates_are_distinct_plans(lg):
    plans = list(tune.candidates(lg))
    assert len(set(plans)) == len(plans)
    for bits, gbits, k16 in plans:
        assert sum(bits) == lg and len(gbits) == len(k16) == len(bits) <= 3
        # the general kernel is asked for only where there is a choice
        assert all(k or p in switchable(bits) for p, k in enumerate(k16)), (bits, k16)


def test_table_header_names_the_passes(tmp_path):
    path = str(tmp_path / "t.txt")
    tune.write_table([(18, 0.35, 0.28, ((8, 10), (4, 4), (1, 1))), (17, 0.139, 0.139, None)], path, 135, 5)
    text = open(path).read()
    assert "10-bit, 9-bit or first 8-bit pass" in text
    assert "18 2 8 10 0 4 4 -1 1 1 0" in text
