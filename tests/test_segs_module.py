"""The native segment tables are an aid: without their module, or with one built
against another torch, the calls go on with the tables made in Python."""

import pytest
import torch

from test1_amd import _native, kernels


@pytest.fixture
def fresh(monkeypatch):
    monkeypatch.setattr(_native, "_segs", None)
    return monkeypatch


def missing(m, tmp_path):
    m.setattr(_native, "SEGS_LIB", str(tmp_path / "none.so"))


def no_library(m, tmp_path):
    (tmp_path / "bad.so").write_bytes(b"not a shared object")
    m.setattr(_native, "SEGS_LIB", str(tmp_path / "bad.so"))


def another_torch(m, tmp_path):
    m.setattr(torch, "__version__", "1.0.0")


@pytest.mark.parametrize("break_it", [missing, no_library, another_torch])
def test_calls_go_on_without_the_module(fresh, tmp_path, break_it):
    break_it(fresh, tmp_path)
    with pytest.warns(RuntimeWarning, match="made in Python"):
        assert _native.segs() is None
    assert _native.segs() is None   # tried once
    # the checks in Python decide, on a host tensor as ever
    with pytest.raises(ValueError, match=r"srcs\[0\] must be a GPU tensor"):
        kernels._list_table([torch.zeros(8, dtype=torch.bfloat16)], "srcs", as_dst=False)
    with pytest.raises(ValueError, match="must be a GPU tensor"):
        kernels.copy_segs_b16([(torch.zeros(8, dtype=torch.bfloat16), torch.zeros(8, dtype=torch.bfloat16))])


def test_the_built_module_loads(fresh):
    assert _native.segs() is not None and _native.segs().TORCH_VERSION == torch.__version__
