"""Lanes that share an entry of a block product must not sum longer chains than
lanes with an entry of their own: the rounding error of the FP32 block of 8
(two lanes to a row of x) against the FP64 product stays that of the block of 2
(one lane).  Chains twice as long raise it by 13 % here; the errors of two
widths differ by about 1 % otherwise, so 5 % tells them apart."""
import numpy as np
import pytest

import lsamd
from lsamd import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [24, 28])
def test_wide_blocks_round_like_narrow_ones(engine, n):
    S = lsamd.Symmetries([lsamd.Symmetry(g, 0) for g in (models.chain_translation(n), models.chain_parity(n))])
    basis = lsamd.DeviceBasis(n, n // 2, 1, S)
    basis.build()
    op = lsamd.DeviceOperator(basis, models.j1j2_chain(n))
    op.build_csr(96)
    x = np.random.default_rng(n).standard_normal((basis.number_states, 8)).astype(np.float32)
    want = np.stack([op.matvec(x[:, q].astype(np.float64), "csr") for q in range(8)], axis=1)

    def error(columns):
        got = np.concatenate([op.matvec_block(np.ascontiguousarray(x[:, q:q + columns]), 32)
                              for q in range(0, 8, columns)], axis=1)
        return np.linalg.norm(got - want) / np.linalg.norm(want)

    narrow, wide = error(2), error(8)
    print(n, narrow, wide, flush=True)
    assert wide <= 1.05 * narrow
