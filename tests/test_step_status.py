"""The decode step's status words (cache.py): counters read as differences.  On the CPU, with the
counts written as the kernels add them."""
import torch


def _engine(layers=2):
    from llm_kvcache_quantization_amd import INT8KVCache

    return INT8KVCache(layers, device="cpu")


def _ptr_row(c, layer):
    c._step_status_ptr(layer, torch.device("cpu"))
    return c._step_status[layer]


def test_clear_drops_counts_of_a_step_that_raised():
    """A step can raise after its append was enqueued (the attention is refused): its flags and
    counts were never pending, and clear() drops them with the rest."""
    c = _engine()
    row = _ptr_row(c, 0)
    row += torch.tensor([1, 40, 0, 7], dtype=torch.int32)  # appended, then the call raised
    c.clear()
    row = _ptr_row(c, 0)
    row[3] += 2
    c._defer_status(0, 1000, "INT8", "[-127, 127]")
    c.flush_status()  # raises ValueError if the stale NaN flag is still there
    assert c._step_seen[0] == row.tolist()


def test_flag_of_another_layers_raised_step_is_cleared_by_a_read():
    c = _engine()
    _ptr_row(c, 1)[2] = 1  # layer 1's step raised after its append
    _ptr_row(c, 0)
    c._defer_status(0, 1000, "INT8", "[-127, 127]")
    c.flush_status()
    _ptr_row(c, 1)
    c._defer_status(1, 1000, "INT8", "[-127, 127]")  # the last layer: read here
    assert c._step_pending == []


def test_counts_are_differences_and_wrap():
    from llm_kvcache_quantization_amd.cache import _since

    assert _since([0, 5, 0, 9], [0, 2, 0, 9]) == [0, 3, 0, 0]
    assert _since([0, -2 ** 31 + 1, 1, 0], [0, 2 ** 31 - 1, 0, 0]) == [0, 2, 1, 0]
