import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "qwen3-image21_amd")
ORACLE = os.path.join(ROOT, "oracle")
for p in (ROOT, PKG, ORACLE, os.path.join(ROOT, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built libqimm.so")


@pytest.fixture(scope="session")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="session")
def qctx(torch_cuda):
    import qimm
    ctx = qimm.Context(0)
    yield ctx
    torch_cuda.cuda.synchronize()
    ctx.close()


@pytest.fixture(scope="session")
def qctx_codes(torch_cuda):
    """A context whose quantized weights keep their codes alone: the decoding kernels take
    every product, as on a card without room for bf16 rows."""
    import qimm
    ctx = qimm.Context(0)
    ctx.set_bf16_rows(qimm.BF16_ROWS_NEVER)
    yield ctx
    torch_cuda.cuda.synchronize()
    ctx.close()
