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
