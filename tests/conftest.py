import importlib.util
import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))


def load_package():
    name = "flash_attn_rtx5060_amd"
    if name in sys.modules:
        return sys.modules[name]
    spec = importlib.util.spec_from_file_location(name, os.path.join(REPO, "flash-attn-rtx5060_amd", "__init__.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def fa():
    return load_package()


@pytest.fixture(scope="session")
def oracle():
    import oracle_binding
    return oracle_binding


@pytest.fixture(params=["alone", "among_others"])
def forward(request, fa):
    """flash_attention_forward of a small problem as it is, which the kernel of 32-row blocks may run, and among copies of itself, which the
    tile kernels do."""
    import functools
    from parity_util import forward_among_others
    return fa.flash_attention_forward if request.param == "alone" else functools.partial(forward_among_others, fa)
