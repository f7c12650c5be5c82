"""The row-batched GEMMs whose products come from the matrix cores
(k_mgemm): sizes that are no multiple of any tile in rows, outputs or K,
weights with signed zeros and products that flush to zero.  Every row must
have the bits of the vector-unit kernel (CIS2_BGEMM16=0) and of the oracle;
the arithmetic is pinned, so there is no tolerance."""
import os

import numpy as np
import pytest

import _oracle as O
from cis2amd import Cis2Model, artifacts

pytestmark = pytest.mark.gpu

ODD = artifacts.ModelSpec("odd", 132, 268, 1, 6, 2, 301, 1e-5, 10000.0, True, head_dim=22)
# K = 20 (one partial group of 16 and one of 4), a vocabulary of many tiles
WIDE = artifacts.ModelSpec("wide-vocab", 20, 28, 1, 2, 1, 40003, 1e-5, 10000.0, True)


class EdgeWeights(artifacts.Weights):
    """The seeded weights with one entry in 16 replaced by +-0 and one in 16
    by +-2^-125 (times an activation below 1/2: a product that is flushed)."""

    def __init__(self, spec, seed):
        super().__init__(spec, seed)
        rng = np.random.default_rng(seed)
        for name, _, arr in self.tensors:
            if not name.endswith("norm.weight"):
                k = rng.integers(0, 16, arr.size)
                arr[k == 0] &= 0x8000
                arr[k == 1] = (arr[k == 1] & 0x8000) | 0x0100


def run(m, n, per_seq, tok, mode):
    os.environ["CIS2_BGEMM16"] = mode
    try:
        i = np.arange(n)
        lg, am = m.forward_rows(i // per_seq, i % per_seq, tok)
    finally:
        del os.environ["CIS2_BGEMM16"]
    return lg.view(np.uint32), am


@pytest.mark.parametrize("spec,n,per_seq", [
    (WIDE, 5, 5),        # LM head: 64 x 16 tiles, one partial
    (WIDE, 16, 4),
    (WIDE, 17, 17),      # the first row count of the 32 x 32 tiles
    (ODD, 931, 19),      # 32 x 32 tiles, the last with 3 rows
    (ODD, 16001, 40),    # 64 x 64 tiles, the last with one row
], ids=lambda v: getattr(v, "name", str(v)))
def test_rows_matrix_core_gemm_bits(spec, n, per_seq):
    w = EdgeWeights(spec, 11)
    nseq = (n + per_seq - 1) // per_seq
    m = Cis2Model(spec, w, max_pos=per_seq, max_seqs=nseq)
    tok = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    lg, am = run(m, n, per_seq, tok, "1")
    lv, av = run(m, n, per_seq, tok, "0")
    assert np.array_equal(lg, lv)
    assert np.array_equal(am, av)
    for s in (0, nseq - 1):
        o = O.OracleModel(spec, w, max_pos=per_seq, reduction=0)
        for p in range(min(per_seq, n - s * per_seq)):
            want = o.forward(p, int(tok[s * per_seq + p])).view(np.uint32)
            assert np.array_equal(want, lg[s * per_seq + p]), (s, p)
