"""Descriptor rows of a grouped product (mpsim_amd.engine): every form an operand was
taken in before the addresses of a call's tensors were looked up once per tensor."""
from collections import namedtuple
from collections.abc import Sequence

import pytest
import torch

Place = namedtuple("Place", "tensor offset")


def _op(a, b, c, n=2):
    return dict(A=a, B=b, C=c, m=n, n=n, k=n, lda=n, ldb=n, ldc=n)


def test_operands_as_tensors_pairs_and_named_pairs():
    from mpsim_amd.engine import _gemm_rows
    t = [torch.zeros(16, dtype=torch.complex64) for _ in range(3)]
    at = [x.data_ptr() for x in t]
    rows = _gemm_rows([_op(t[0], (t[1], 4), Place(t[2], 8))])
    assert rows[0][:3] == (at[0], at[1] + 32, at[2] + 64)


class _Lazy(Sequence):
    """Products whose operands are views made when they are asked for (`pairs`: with an
    offset)."""

    def __init__(self, base, count, pairs):
        self.base, self.count, self.pairs = base, count, pairs

    def __len__(self):
        return self.count

    def __getitem__(self, i):
        if i >= self.count:
            raise IndexError
        v = [self.base[12 * i + 4 * j:12 * i + 4 * j + 4] for j in range(3)]
        return _op(*[(x, 0) for x in v] if self.pairs else v)


@pytest.mark.parametrize("pairs", [False, True])
def test_operands_made_on_the_way_have_their_own_addresses(pairs):
    from mpsim_amd.engine import _gemm_rows
    base = torch.zeros(12 * 50, dtype=torch.complex64)
    p = base.data_ptr()
    rows = _gemm_rows(_Lazy(base, 50, pairs))
    assert [r[:3] for r in rows] == [tuple(p + 8 * (12 * i + 4 * j) for j in range(3)) for i in range(50)]
