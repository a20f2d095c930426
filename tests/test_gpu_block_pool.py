"""The device-block pool: reused blocks give the same results, from several
host threads too, and ls_chpl_finalize gives the kept memory back."""
import threading

import numpy as np
import pytest
import torch

import lsamd
from lsamd import models

pytestmark = pytest.mark.gpu


def product(n, seed):
    S = lsamd.Symmetries([lsamd.Symmetry(g, 0) for g in (models.chain_translation(n), models.chain_parity(n))])
    basis = lsamd.DeviceBasis(n, n // 2, 1 if n % 2 == 0 else None, S)
    basis.build()
    operator = lsamd.DeviceOperator(basis, models.j1j2_chain(n))
    operator.build_csr(96)
    x = np.random.default_rng(seed).standard_normal(basis.number_states)
    return operator.matvec(x, "csr")


def test_rebuilds_and_threads_give_the_same_bits(engine):
    sizes = (10, 17, 20, 22)
    first = {n: product(n, n) for n in sizes}
    for n in sizes[::-1] + sizes:
        assert np.array_equal(product(n, n), first[n])
    wrong = []

    def work(n):
        for _ in range(3):
            if not np.array_equal(product(n, n), first[n]):
                wrong.append(n)

    threads = [threading.Thread(target=work, args=(n,)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_finalize_gives_the_memory_back(engine):
    lib = lsamd.load()
    lib.ls_chpl_finalize()
    before = torch.cuda.mem_get_info()[0]
    S = lsamd.Symmetries([lsamd.Symmetry(models.chain_translation(26), 0)])
    basis = lsamd.DeviceBasis(26, 13, 1, S)
    basis.build()
    operator = lsamd.DeviceOperator(basis, models.j1j2_chain(26))
    operator.build_csr(96)
    del operator, basis
    lib.ls_chpl_finalize()
    assert torch.cuda.mem_get_info()[0] >= before - (64 << 20)


def keep_blocks():
    """Blocks of a released operator and basis stay with the engine."""
    lsamd.device_trim()
    free = torch.cuda.mem_get_info()[0]
    product(24, 1)
    return free


def test_trim_gives_the_memory_back(engine):
    free = keep_blocks()
    assert torch.cuda.mem_get_info()[0] < free - (8 << 20)
    assert lsamd.device_trim() > 8 << 20
    assert torch.cuda.mem_get_info()[0] >= free - (8 << 20)
    assert lsamd.device_trim() == 0


def test_a_failing_allocation_empties_the_pool_first(engine):
    free = keep_blocks()
    assert torch.cuda.mem_get_info()[0] < free - (8 << 20)
    with pytest.raises(lsamd.EngineError, match="allocation failed"):
        lsamd.DeviceArray(1 << 50)  # more than any device has
    assert torch.cuda.mem_get_info()[0] >= free - (8 << 20)
    assert np.isfinite(product(16, 1)).all()  # and the engine goes on
