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


def test_a_short_prompt_takes_a_short_prompts_memory(model):
    """Buffers of batched passes come in one allocation sized for the prompt,
    grow with longer ones, are kept for shorter ones and go with the context."""
    d, wide, q, kv, ff = 512, 512, 512, 512, 768
    before = model.get("live")
    c = model.context(2048, 32)
    base = model.get("live")
    model.set("mallocs", 0)
    st, p = model.eval(c, np.arange(9))
    assert st == 0 and np.array_equal(model.row(p), model.want([8])[0])
    assert model.get("mallocs") == 1 and model.get("batches") == 2      # (two layers)
    assert model.get("live") - base <= 64 * 4 * (d + wide + q + 2 * kv + ff + 2) + 8 * 256
    ids = np.arange(300)
    st, p = model.eval(c, ids)
    assert st == 0 and np.array_equal(model.row(p), model.want(ids)[-1])
    assert model.get("mallocs") == 2 and model.get("max_batch") == 300
    st, _ = model.eval(c, np.arange(20))
    assert st == 0 and model.get("mallocs") == 2
    st, _ = model.eval(c, np.arange(600) % 500)
    assert st == 0 and model.get("mallocs") == 2
    model.lib.fox_context_destroy(c)
    assert model.get("live") == before


def test_passes_of_what_memory_there_is(model):
    """Where the buffers of the whole prompt cannot be had: passes of 256, of
    64, and of eight tokens, with the same logits."""
    ids = np.arange(500)
    per = 4 * (512 * 5 + 768 + 2)
    for limit, largest in ((0, 500), (300 * per, 256), (100 * per, 64), (10 * per, 0)):
        c = model.context(512, 32)
        model.set("max_batch", 0)
        model.set("mallocs", 0)
        model.set("fail_above", limit)
        st, p = model.eval(c, ids)
        assert st == 0 and np.array_equal(model.row(p), model.want(ids)[-1])
        assert model.get("max_batch") == largest
        assert model.get("mallocs") == (largest > 0)        # (not tried again at every pass)
        model.set("fail_above", 0)
        model.lib.fox_context_destroy(c)


@pytest.mark.parametrize("n_batch,largest", [(3, 0), (8, 0), (9, 9), (16, 16), (200, 192), (0, 500),
                                             (32, 500), (5000, 500)])
def test_n_batch_bounds_a_pass(model, n_batch, largest):
    """A caller's n_batch bounds the tokens of a pass and its memory (three even
    passes of whole groups of 64 where 200 are allowed); 0 and the default
    leave them to the library."""
    ids = np.arange(500)
    c = model.context(512, n_batch)
    base = model.get("live")
    st, p = model.eval(c, ids)
    assert st == 0 and np.array_equal(model.row(p), model.want(ids)[-1])
    assert model.get("max_batch") == largest
    if 8 < n_batch < 32:
        assert model.get("live") - base <= n_batch * 4 * (512 * 5 + 768 + 2) + 8 * 256
    model.lib.fox_context_destroy(c)


def test_a_pass_without_memory_runs_in_passes_of_eight(model):
    """Batched attention's workspace refused, in the first and in a later pass:
    the same logits through the decode kernels, and no further attempt."""
    for first in (20, 64):
        c = model.context(2048, 64)
        ids = np.arange(first + 40)
        if first == 64:
            assert model.eval(c, ids[:64])[0] == 0
        model.set("max_batch", 0)
        model.set("eights", 0)
        model.fail_attention(1)
        n = 64 if first == 64 else 0
        st, p = model.eval(c, ids[n:])
        assert st == 0 and np.array_equal(model.row(p), model.want(ids)[-1])
        assert model.lib.fox_context_position(c) == len(ids)
        assert model.get("eights") == 2 * -(-(len(ids) - n) // 8)       # (two layers)
        model.set("batches", 0)
        st, p = model.eval(c, ids)
        assert st == 0 and model.get("batches") == 0
        model.lib.fox_context_destroy(c)


def test_logits_rows_without_memory(model):
    """fox_eval_all's block of logits rows refused: every row all the same."""
    c = model.context(256, 32)
    assert model.eval(c, np.arange(100))[0] == 0                         # (the pass's buffers)
    model.set("fail_above", 64 * 600 * 4 - 1)
    ids = np.arange(100) + 3
    st, got = model.eval_all(c, ids)
    assert st == 0 and np.array_equal(got, model.want(ids))
    assert model.lib.fox_context_position(c) == 200
    model.lib.fox_context_destroy(c)


def test_few_tokens_on_a_long_cache_attend_in_eights(model):
    """The batched attention kernels run a token's sums in one lane: few tokens
    on a long cache take the decode kernels' attention inside a batched pass."""
    c = model.context(32768, 32)
    for pos, n, eights in ((0, 9, 0), (0, 300, 0), (200, 12, 0), (1024, 9, 2), (8192, 24, 3),
                           (8192, 64, 0), (30000, 32, 4), (30000, 300, 0)):
        assert model.lib.fox_context_set_position(c, pos) == 0
        model.set("small_attn", 0)
        model.set("batches", 0)
        ids = np.arange(n)
        st, p = model.eval(c, ids)
        assert st == 0 and np.array_equal(model.row(p), model.want(ids)[-1])
        assert model.get("small_attn") == 2 * eights, (pos, n)          # (two layers)
        assert model.get("batches") == 2
    model.lib.fox_context_destroy(c)
