"""fox_eval's own decisions, on the CPU over a stub of the device library
(host_stub.py)."""
import numpy as np
import pytest

from host_stub import StubModel, build


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return build(str(tmp_path_factory.mktemp("stub")))


@pytest.fixture
def model(lib, tmp_path):
    m = StubModel(lib, str(tmp_path / "m.gguf"))
    yield m
    m.close()


@pytest.mark.parametrize("n", [3, 20])
def test_eval_all_leaves_the_logits_of_eval(model, n):
    """The row that fox_eval handed out is fox_eval's: a later fox_eval_all
    writes to its caller's memory only."""
    c = model.context(128, 32)
    st, p = model.eval(c, [7, 9])
    assert st == 0 and np.array_equal(model.row(p), model.want([9])[0])
    ids = np.arange(100, 100 + n)
    st, got = model.eval_all(c, ids)
    assert st == 0 and np.array_equal(got, model.want(ids))
    assert np.array_equal(model.row(p), model.want([9])[0])
    model.lib.fox_context_destroy(c)
