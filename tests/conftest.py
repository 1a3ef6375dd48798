import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "tests"), os.path.join(ROOT, "tests", "golden")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device); run with -m gpu")
    config.addinivalue_line("markers", "slow: long statistical runs")


@pytest.hookimpl(hookwrapper=True)
def pytest_pyfunc_call(pyfuncitem):
    """A test that asks for the reference build where it does not exist (it is made from the reference's sources) is
    skipped, as the tests that look for it first are."""
    outcome = yield
    error = outcome.excinfo[1] if outcome.excinfo else None
    if isinstance(error, RuntimeError) and "missing (built only where the reference sources are present)" in str(error):
        outcome.force_exception(pytest.skip.Exception(str(error)))


@pytest.fixture(scope="session")
def golden():
    import json
    with open(os.path.join(ROOT, "tests", "golden", "golden.json")) as f:
        return json.load(f)
