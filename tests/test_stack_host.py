"""What the stack keeps between calls, as far as it shows without a GPU: copies, files, replicas."""
import copy
import ctypes
import io
import pickle

import pytest
import torch

from layers import MvpaKVCache
from models.mvpformer import MVPFormerConfig, MVPFormerModel, _StackOperands


def _model(**kw):
    torch.manual_seed(0)
    dims = dict(n_positions=8, n_channels=6, n_embd=64, n_layer=2, n_head=2, n_head_kv=1, n_inner=64)
    dims.update(kw)
    return MVPFormerModel(MVPFormerConfig(**dims)).eval()


def _capsule():
    """What watch and plans are to Python: an opaque pointer that neither copies nor pickles."""
    new = ctypes.pythonapi.PyCapsule_New
    new.restype, new.argtypes = ctypes.py_object, (ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p)
    return new(1, None, None)


def _through_file(model):
    buf = io.BytesIO()
    torch.save(model, buf)
    buf.seek(0)
    return torch.load(buf, weights_only=False)


@pytest.mark.parametrize("how", [copy.copy, copy.deepcopy, lambda m: pickle.loads(pickle.dumps(m)), _through_file],
                         ids=["copy", "deepcopy", "pickle", "save"])
def test_a_model_with_a_plan_is_copied(how):
    model = _model()
    model._stack = _StackOperands()
    model._stack.watch = _capsule()
    other = how(model)
    assert other._stack is None and model._stack is not None
    assert all(torch.equal(a, b) for a, b in zip(model.state_dict().values(), other.state_dict().values()))


def test_a_model_saved_without_plans_loads():
    model = _model()
    state = {n: v for n, v in model.__getstate__().items() if n != "_stack"}
    other = MVPFormerModel.__new__(MVPFormerModel)
    other.__setstate__(state)
    assert other._stack is None


def test_a_replica_has_no_plan():
    model = _model()
    model._stack = _StackOperands()
    model._stack.watch = _capsule()
    replica = model._replicate_for_data_parallel()
    assert replica._stack is None and model._stack is not None


@pytest.mark.parametrize("max_steps,slack", [(1, 0), (3, 0), (3, 1), (4, 2)])
def test_a_cache_counts_a_step_once_it_is_written(max_steps, slack):
    """next_slot() names make_room()'s slot and changes nothing; a step that is never counted costs a full
    window its oldest step and nothing else, however often it is tried."""
    cache = MvpaKVCache(1, 1, 1, 4, max_steps, dtype=torch.float32, device="cpu", slack=slack)
    cache.k.zero_()                                                   # so that it can be compared with itself
    held = []
    for step in range(4 * max_steps + 7):
        before = (cache.start, cache.length, cache.k.clone())
        slot = cache.next_slot()
        assert (cache.start, cache.length) == before[:2] and torch.equal(cache.k, before[2])
        for _ in range(1 + step % 2):                                 # tried again where a step did not come about
            assert cache.make_room() == cache.next_slot() == slot
            assert cache.views()[0][0, 0, :, 0, 0].tolist() == held[max(0, len(held) - max_steps + 1):]
        cache.append(*(torch.full((1, 1, 1, 4), float(step)) for _ in range(2)))
        held = (held + [float(step)])[-max_steps:]
        assert cache.views()[0][0, 0, :, 0, 0].tolist() == held
