import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP path)")


def pytest_collection_modifyitems(items):
    """The tests that fail where the compiled reference (oracle/_ref) was not built, for want of its sources,
    run last there: a run that stops at its first failure has then run all the others."""
    import oracle_ctypes as oc

    if os.path.exists(oc.REF_SO) and os.path.exists(oc.REF_MI355X_SO):
        return

    def needs_reference(item):
        module = os.path.basename(str(item.path))
        return module in ("test_dropin_gpu.py", "test_module_ops_gpu.py") or (
            module == "test_generate_gpu.py" and item.name.startswith("test_reference_"))

    items.sort(key=needs_reference)


@pytest.fixture(autouse=True)
def _release_device_buffers():
    yield
    import gpu_util

    gpu_util.release_all()
