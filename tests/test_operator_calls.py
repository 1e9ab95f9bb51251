"""Calls of the operator that reach the native code without a Python frame take their arguments as the functions they stand for
do (by position and by name, with the defaults), are bound, inspected and kept as those are, and give way to whatever a user puts
in their place."""

import inspect
import sys
import types
import weakref

import pytest
import torch

from pplx_garden_amd.kernels.p2p_all_to_all import P2PAllToAll, _call_without_a_frame
from pplx_garden_amd.native import p2p_all_to_all as native


@pytest.fixture()
def world():
    module = native.load_extension()
    _call_without_a_frame(module)
    context = module.Context(0, 2)     # (closed: nothing is launched)

    def make(cls, rank):
        op = cls.__new__(cls)
        op._all_to_all = None
        op._operator = module.Operator(context, rank, 1, 128, 1, 2, 4, torch.float8_e4m3fn, torch.bfloat16, True, -1)
        return op

    dispatch = dict(out_expert_num_tokens=torch.zeros(2, dtype=torch.int32),
                    out_expert_x=torch.zeros((8, 128), dtype=torch.float8_e4m3fn), out_expert_x_scale=torch.zeros((8, 1)),
                    dp_x=torch.zeros((5, 128), dtype=torch.bfloat16), dp_x_scale=None,
                    indices=torch.zeros((5, 4), dtype=torch.int32).view(torch.uint32), weights=torch.zeros((5, 4)))
    combine = dict(out_tokens=torch.zeros((5, 128), dtype=torch.bfloat16), indices=dispatch["indices"],
                   weights=dispatch["weights"], expert_y=torch.zeros((8, 128), dtype=torch.bfloat16))
    return context, make, dispatch, combine


def test_arguments_by_name_by_position_and_by_default(world):
    context, make, d, c = world
    for args, kwargs in [((), d), (tuple(d.values()), {}), (tuple(d.values())[:3], dict(list(d.items())[3:])),
                         ((), dict(reversed(list(d.items())), do_recv=True, bound_m=None)),
                         ((), {"".join(list(k)): v for k, v in d.items()})]:      # (names that are not interned)
        op = make(P2PAllToAll, 0)
        assert op.dispatch(*args, **kwargs) is None and context.pending("dispatch") == 1
        with pytest.raises(RuntimeError, match="destroyed"):
            make(P2PAllToAll, 1).dispatch(**d)
        assert context.pending("dispatch") == 0
    op = make(P2PAllToAll, 0)
    assert op.combine(**c) is None and context.pending("combine") == 1
    with pytest.raises(RuntimeError, match="same expert_y dtype and accumulate"):
        make(P2PAllToAll, 1).combine(**c, accumulate=True)
    with pytest.raises(RuntimeError, match="destroyed"):      # do_send alone runs at once
        op.dispatch(**d, do_send=True, do_recv=False)
    with pytest.raises(AssertionError):
        op.dispatch(**d, do_send=False, do_recv=False)


@pytest.mark.parametrize("halves", [{}, dict(do_recv=False), dict(do_send=False)])
@pytest.mark.parametrize("name", ["dispatch", "combine"])
def test_a_method_taken_before_destroy_refuses_calls_after_it(world, name, halves):
    context, make, d, c = world
    op = make(P2PAllToAll, 0)
    held = getattr(op, name)
    op._operator = None     # as destroy() leaves it
    with pytest.raises(AssertionError):
        held(**(d if name == "dispatch" else c), **halves)
    assert context.pending(name) == 0


@pytest.mark.parametrize("name", ["dispatch", "combine"])
def test_a_method_is_the_functions_bound_to_the_operator(world, name):
    _, make, _, _ = world
    op = make(P2PAllToAll, 0)
    method, function = getattr(op, name), getattr(P2PAllToAll, name)
    assert isinstance(method, types.MethodType) and method.__self__ is op and method.__func__ is function
    assert list(inspect.signature(method).parameters) == list(inspect.signature(function).parameters)[1:]
    assert inspect.signature(method).parameters["do_recv"].default is True
    assert method.__annotations__["weights"] and weakref.WeakMethod(method)() == method
    alive = weakref.ref(op)
    del op
    assert alive() is not None      # kept by the bound method


def test_profilers_see_the_function_and_other_code_of_it_runs(world, monkeypatch):
    context, make, d, c = world
    seen = []
    sys.setprofile(lambda frame, event, arg: seen.append(frame.f_code) if event == "call" else None)
    try:
        make(P2PAllToAll, 0).dispatch(**d)
    finally:
        sys.setprofile(None)
    assert P2PAllToAll.dispatch.__code__ in seen and context.pending("dispatch") == 1
    monkeypatch.setattr(P2PAllToAll.combine, "__defaults__", (None, False, False, False))
    with pytest.raises(AssertionError, match="do_send || do_recv"):
        make(P2PAllToAll, 0).combine(**c)
    monkeypatch.undo()
    assert make(P2PAllToAll, 0).combine(**c) is None and context.pending("combine") == 1


@pytest.mark.parametrize("args,kwargs,match", [
    ((), dict(unknown=1), "unexpected keyword"), ((torch.zeros(2, dtype=torch.int32),), {}, "multiple values"),
    (tuple(range(11)), None, "11 were given"), ((), None, "missing required argument: 'out_expert_num_tokens'")])
def test_wrong_arguments_are_type_errors(world, args, kwargs, match):
    _, make, d, _ = world
    with pytest.raises(TypeError, match=match):
        make(P2PAllToAll, 0).dispatch(*args, **({} if kwargs is None else {**d, **kwargs}))


def test_the_class_keeps_its_functions_and_users_their_replacements(world, monkeypatch):
    context, make, d, _ = world
    assert isinstance(P2PAllToAll.dispatch, types.FunctionType)
    assert list(inspect.signature(P2PAllToAll.combine).parameters)[-1] == "accumulate"

    class Counting(P2PAllToAll):
        calls = 0

        def dispatch(self, *args, **kwargs):
            self.calls += 1
            return super().dispatch(*args, **kwargs)

    op = make(Counting, 0)
    assert op.dispatch(**d) is None and op.calls == 1 and context.pending("dispatch") == 1
    op = make(P2PAllToAll, 1)
    op._operator = None     # as destroy() leaves it
    with pytest.raises(AssertionError):
        op.dispatch(**d)
    monkeypatch.setattr(P2PAllToAll, "dispatch", lambda self, **kwargs: "replaced")
    _call_without_a_frame(native.load_extension())
    assert make(P2PAllToAll, 0).dispatch(**d) == "replaced"
