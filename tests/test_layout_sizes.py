"""Sizes of the degree blocks, which the launch rules of the factor rest on: blocks
of one parity are of one size, and no block has more than four times another's rows."""
import itertools

import pytest


def _blocks(m, lmax, symm, symmB0, fields, N1):
    from kore_amd import backend
    try:
        backend.lib()
    except backend.KoreLibraryError as e:       # pragma: no cover
        pytest.skip(str(e))
    return backend.layout_blocks(backend.make_layout(m, lmax, symm, N1, *fields, symmB0=symmB0))


@pytest.mark.parametrize("m", [0, 1, 2, 5])
@pytest.mark.parametrize("symm", [1, -1])
@pytest.mark.parametrize("symmB0", [1, -1])
def test_blocks_of_one_parity_have_one_size(m, symm, symmB0):
    for fields in itertools.product([0, 1], repeat=4):      # hydro, magnetic, thermal, compositional
        if not any(fields):
            continue
        for nl, N1 in itertools.product([2, 4, 10], [1, 7, 64]):
            n, sizes, order = _blocks(m, m + nl - 1, symm, symmB0, fields, N1)
            assert sum(sizes) == n == len(set(order))
            for parity in (0, 1):
                assert len(set(sizes[parity::2])) <= 1, (fields, list(sizes))
            assert max(sizes) <= 4 * min(sizes), (fields, list(sizes))
