"""The device memory that a system of a batch is charged with.

A server admits requests by orr_batch_bytes_bound, so a request that fits a given
budget must go on fitting it: the bounds may shrink, not grow.
"""
import pytest

import orrery_amd as E


def bound(n, solver, quadrupole=False):
    return E.DeviceBatch.bytes_bound([E.BatchSystem(n, 0.01, 1e-3, solver=solver)],
                                     E.BatchConfig(quadrupole=quadrupole))


@pytest.mark.parametrize("n,most", [
    (256, 162136), (1000, 502836), (4095, 1884006), (4096, 1884240), (10000, 6471504), (16384, 13916376),
    (16385, 14637356), (32768, 46130232), (32769, 46886344), (65536, 155515640), (131071, 564602626),
    (262144, 2144043896)])
def test_direct_system_bound(n, most):
    assert bound(n, 0) <= most


@pytest.mark.parametrize("n,quadrupole,most", [
    (256, False, 295905), (256, True, 357405), (1000, False, 975315), (1000, True, 1201515),
    (4096, False, 3414502), (4096, True, 4332502), (16384, False, 14053447), (16384, True, 17718547),
    (16385, False, 14243740), (16385, True, 17908940), (32768, False, 30532468), (32769, True, 37559301),
    (60000, False, 55757119), (60000, True, 69172419), (100000, False, 92779655), (131071, True, 150840385),
    (262144, False, 242877579), (262144, True, 301478379), (2097152, True, 2387037417)])
def test_tree_system_bound(n, quadrupole, most):
    assert bound(n, 1, quadrupole) <= most
