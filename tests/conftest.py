import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "flash-attention_amd")
for p in (ROOT, PKG):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(autouse=True)
def _no_row_orders_of_other_tests():
    """Row orders of block layouts are kept by the address of the converted mask; one left by another test's mask at the same address is a valid
    order, but another one, and moves the last bits of a result that a test compares exactly (by up to 2.4e-4 in fp16)."""
    mod = sys.modules.get("flash_attn.flash_blocksparse_attn_interface")
    if mod is not None:
        mod._ROW_ORDERS.clear()


@pytest.fixture(scope="session")
def lib():
    """The C-ABI library, built in-tree beforehand; built here only if nothing is there."""
    from flash_attn import flash_attn_gfx950 as be
    if not os.path.exists(be.LIB_PATH):
        sys.path.insert(0, PKG)
        import build as _build
        _build.build()
    return be.load_library()
