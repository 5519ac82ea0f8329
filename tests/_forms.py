"""The encode kernels a test can force, by head dim (the `form` fixture of
conftest.py sets the environment, which is read at every call)."""
import pytest

KERNELS = {64: ["wide", "split16", "split32", "exact"], 128: ["wide", "split16", "split32"],
           256: ["d256"]}


def encode_forms(*dims):
    """Parametrises `form`, the head dim, over the kernels that serve these dims."""
    params = [(k, D) for D in dims for k in KERNELS[D]]
    return pytest.mark.parametrize("form", params, indirect=True,
                                   ids=[f"{k}-{D}" for k, D in params])
