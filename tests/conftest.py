import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fame-isotropic-gpu_amd", "python"))
sys.path.insert(0, os.path.join(ROOT, "oracle"))
sys.path.insert(0, os.path.join(ROOT, "tests"))

# an empty reference directory is no reference tree: what is compared with its files is skipped
_REF = "/root/reference"
if "FAME_REFERENCE_DIR" not in os.environ and os.path.isdir(_REF) and not os.listdir(_REF):
    os.environ["FAME_REFERENCE_DIR"] = os.path.join(ROOT, "no-reference-tree")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP path through the C-ABI)")
    config.addinivalue_line("markers", "slow: longer CPU checks")


@pytest.fixture(scope="session")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)
