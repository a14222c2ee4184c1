"""The rule behind the pair loads of the group-order kernel: of the suffix parents of a sorted tuple,
the next tuple's are the next entries for every dropped position except the first one in which the
two tuples differ; that one is unchanged when the last position differs."""
import itertools

import pytest


@pytest.mark.parametrize("suf", [4, 5])
@pytest.mark.parametrize("m", [1, 2, 3, 5, 8])
def test_parents_of_the_next_tuple(m, suf):
    shorter = {t: i for i, t in enumerate(itertools.combinations_with_replacement(range(m), suf - 1))}
    tuples = list(itertools.combinations_with_replacement(range(m), suf))
    for a, b in zip(tuples, tuples[1:]):
        e = next(j for j in range(suf) if a[j] != b[j])
        for j in range(suf):
            pa, pb = shorter[a[:j] + a[j + 1:]], shorter[b[:j] + b[j + 1:]]
            if j != e:
                assert pb == pa + 1, (a, b, j)
            elif e == suf - 1:
                assert pb == pa, (a, b)
            # the pair load reads the entry after a's parent in every case. It is past the parents of
            # this block only for a = (x, m-1, .., m-1) without x, and then the block's prefix ends
            # below m - 1 (at most x), so that another block follows in the layer
            assert pa + 1 < len(shorter) or (j == e == 0 and a[0] < m - 1), (a, b, j)
