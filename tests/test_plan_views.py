"""The C views a plan keeps (plan build and attention launch) follow a buffer or configuration
that is put in another's place, the attention's also one whose storage is replaced in the tensor itself,
and the attention's arguments take any object with a plan's fields.  A copied plan makes its own."""
import copy
import pickle
import types

import pytest
import torch

from sglang_decode.config import DecodeConfig
from sglang_decode.kernels.attention import plan_args
from sglang_decode.runtime.workspace import PlanBuffers


@pytest.mark.parametrize("field", ["lengths", "mode", "order", "static_head"])
def test_views_follow_replaced_buffers(field):
    c = DecodeConfig(batch_capacity=4, max_splits=2, max_context=256)
    plan = PlanBuffers(c, "cpu")
    plan.c_struct(), plan.decode_args()
    other = getattr(plan, field).clone()
    setattr(plan, field, other)
    assert getattr(plan.c_struct(), field) == other.data_ptr()
    assert getattr(plan.decode_args(), field) == other.data_ptr()
    plan.config = DecodeConfig(batch_capacity=4, max_splits=2, max_context=256, workers=7)
    assert plan.decode_args().workers == 7
    lookalike = types.SimpleNamespace(**{k: v for k, v in vars(plan).items() if not k.startswith("_")})
    assert bytes(plan_args(lookalike)) == bytes(plan.decode_args())


@pytest.mark.parametrize("field", ["lengths", "mode", "order", "static_next"])
def test_arguments_follow_storage_replaced_in_place(field):
    plan = PlanBuffers(DecodeConfig(batch_capacity=4, max_splits=2, max_context=256), "cpu")
    plan.decode_args()
    tensor = getattr(plan, field)
    for change in (lambda: tensor.set_(tensor.clone()), lambda: setattr(tensor, "data", tensor.clone())):
        before = tensor.data_ptr()
        change()
        assert tensor.data_ptr() != before and getattr(plan.decode_args(), field) == tensor.data_ptr()
    assert bytes(plan_args(plan)) == bytes(plan.decode_args())


def test_a_wrapper_keeps_the_fields_it_replaces(monkeypatch):
    """An object that hands everything but some fields of its own on to a plan: the launch takes those fields."""
    from sglang_decode.kernels import attention as A

    class Wrapper:
        def __init__(self, plan):
            self.plan, self.lengths = plan, plan.lengths.clone()

        def __getattr__(self, name):
            return getattr(self.plan, name)

    seen = []

    class Library:
        def sgd_persistent_decode(self, args, stream):
            seen.append(args._obj.lengths)
            return 0

        def sgd_attention_kernel(self, args):
            return 1

    monkeypatch.setattr(A._lib, "lib", lambda: Library())
    monkeypatch.setattr(A._lib, "stream_handle", lambda device: 0)
    plan = PlanBuffers(DecodeConfig(batch_capacity=4, max_splits=2, max_context=256), "cpu")
    wrapper, x = Wrapper(plan), torch.zeros((4, 32, 128), dtype=torch.bfloat16)
    layer = types.SimpleNamespace(counter=x, partial=x, lse=x, output=x)
    for p in (plan, wrapper):
        A.persistent_decode(p, layer, x, x, x, x, None, 1.0, (1,) * 4, (1,) * 4, (1, 1), False)
    assert seen == [plan.lengths.data_ptr(), wrapper.lengths.data_ptr()]


def test_a_launched_plan_copies_and_pickles():
    plan = PlanBuffers(DecodeConfig(batch_capacity=4, max_splits=2, max_context=256), "cpu")
    plan.c_struct(), plan.decode_args()
    plan.lengths.fill_(7)
    for other in (copy.deepcopy(plan), pickle.loads(pickle.dumps(plan))):
        assert torch.equal(other.arena, plan.arena) and other.config == plan.config
        assert other.decode_args().lengths == other.lengths.data_ptr() != plan.lengths.data_ptr()
        assert other.c_struct().lengths == other.lengths.data_ptr()


def test_each_launch_has_its_own_arguments():
    plan = PlanBuffers(DecodeConfig(batch_capacity=4, max_splits=2, max_context=256), "cpu")
    a = plan.decode_args()
    a.q, a.workers = 64, 1
    assert plan.decode_args().q is None and plan.decode_args().workers == plan.config.workers
