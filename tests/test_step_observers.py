"""``step()`` outside torch's profiler range unless something would see it.

The range, and torch's global and per-optimizer step hooks, come from the
wrapper torch puts around every optimizer's step; an unobserved step leaves
it out.
"""

from __future__ import annotations

import functools
import warnings

import pytest
import torch
from torch.optim.optimizer import register_optimizer_step_post_hook, register_optimizer_step_pre_hook
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from sr_states import _group_walk
from sr_states.optim._state import StateOptimizer


class Counting(StateOptimizer):
    _state_names = ("momentum_buffer",)

    def __init__(self, params):
        super().__init__(params, {"lr": 0.1})
        self.updates = 0

    def _step_group(self, group, formats, items, rng_step):
        assert not torch.is_grad_enabled()
        self.updates += 1


class Overriding(Counting):
    def step(self, closure=None):
        return super().step(closure)


def _optimizer(cls=Counting):
    return cls([torch.nn.Parameter(torch.zeros(3))])


def test_a_plain_step_runs_once_and_returns_the_closure_loss():
    optimizer = _optimizer()
    assert not optimizer._step_observed()
    assert optimizer.step(lambda: torch.tensor(2.0, requires_grad=True) * 3) == 6.0
    assert optimizer.updates == 1 and torch.is_grad_enabled()


@pytest.mark.parametrize("cls", [Counting, Overriding])
def test_step_hooks_run_once_and_may_replace_the_arguments(cls):
    optimizer, seen = _optimizer(cls), []
    handles = [
        register_optimizer_step_pre_hook(lambda o, args, kwargs: seen.append("global pre")),
        register_optimizer_step_post_hook(lambda o, args, kwargs: seen.append("global post")),
        optimizer.register_step_pre_hook(lambda o, args, kwargs: ((o, lambda: 5.0), {})),
        optimizer.register_step_post_hook(lambda o, args, kwargs: seen.append("post")),
    ]
    try:
        assert optimizer.step() == 5.0
    finally:
        for handle in handles:
            handle.remove()
    assert sorted(seen) == ["global post", "global pre", "post"] and optimizer.updates == 1
    optimizer.step()
    assert len(seen) == 3 and optimizer.updates == 2


def test_a_profiler_sees_the_step_range():
    optimizer = _optimizer()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        assert _group_walk.observed()
        optimizer.step()
    assert any(event.key == "Optimizer.step#Counting.step" for event in profile.key_averages())
    assert not _group_walk.observed()


def test_a_dispatch_mode_counts_as_an_observer():
    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert _group_walk.observed()
    assert not _group_walk.observed()


def test_a_scheduler_still_tracks_the_step():
    optimizer = _optimizer()
    scheduler = torch.optim.lr_scheduler.StepLR(optimizer, 1)
    optimizer.step()
    scheduler.step()
    assert optimizer.updates == 1


@pytest.mark.parametrize("call,positional,named", [
    (lambda o, f: o.step(), 0, ()),
    (lambda o, f: o.step(None), 1, ()),
    (lambda o, f: o.step(f), 1, ()),
    (lambda o, f: o.step(closure=f), 0, ("closure",)),
])
def test_step_hooks_see_the_call_as_it_was_made(call, positional, named):
    optimizer, seen = _optimizer(), []
    optimizer.register_step_pre_hook(lambda o, args, kwargs: seen.append((args[0] is o, len(args), tuple(kwargs))))
    optimizer.register_step_post_hook(lambda o, args, kwargs: seen.append((args[0] is o, len(args), tuple(kwargs))))
    call(optimizer, lambda: 2.0)
    assert seen == [(True, 1 + positional, named)] * 2 and optimizer.updates == 1


def test_a_pre_hook_may_add_the_closure_by_name():
    optimizer = _optimizer()
    optimizer.register_step_pre_hook(lambda o, args, kwargs: (args, {**kwargs, "closure": lambda: 5.0}))
    assert optimizer.step() == 5.0 and optimizer.updates == 1


def test_a_subclass_may_use_the_name_of_an_inner_step():
    optimizer = _optimizer()
    optimizer._step = 0
    optimizer.step()
    assert optimizer.updates == 1 and optimizer._step == 0


def _patched_after_construction(base):
    class Patched(base):
        pass

    optimizer, inherited = _optimizer(Patched), Patched.step

    @functools.wraps(inherited)
    def step(self, *args, **kwargs):
        return inherited(self, *args, **kwargs)

    Patched.step = step
    return optimizer


def _patched_before_construction(base):
    class Patched(base):
        pass

    @functools.wraps(Patched.step)
    def step(self, *args, **kwargs):
        return base.step(self, *args, **kwargs)

    Patched.step = step
    return _optimizer(Patched)


def _override_named_like_the_inherited(base):
    class Override(base):
        @functools.wraps(base.step)
        def step(self, closure=None):
            return super().step(closure)

    return _optimizer(Override)


def _override_named_like_the_base(base):
    class Override(base):
        @functools.wraps(StateOptimizer.step)
        def step(self, closure=None):
            return super().step(closure)

    return _optimizer(Override)


@pytest.mark.parametrize("constructed", [False, True])
@pytest.mark.parametrize("make", [_patched_after_construction, _patched_before_construction,
                                  _override_named_like_the_inherited, _override_named_like_the_base])
def test_patched_and_wrapped_steps_keep_hooks_and_range(make, constructed):
    class Base(Counting):
        pass

    if constructed:  # torch has wrapped the base class's step, and marked it as wrapped
        _optimizer(Base)
    optimizer, seen = make(Base), []
    optimizer.register_step_pre_hook(lambda *a: seen.append("pre"))
    optimizer.register_step_post_hook(lambda *a: seen.append("post"))
    optimizer.step()
    assert seen == ["pre", "post"] and optimizer.updates == 1
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        optimizer.step()
    assert sum(event.key.startswith("Optimizer.step#") for event in profile.key_averages()) == 1


def test_a_step_within_a_step_has_hooks_of_its_own():
    optimizer, seen = _optimizer(Overriding), []
    optimizer.register_step_post_hook(lambda o, args, kwargs: seen.append(o.updates))
    optimizer.step(lambda: optimizer.step())
    assert seen == [1, 2]
    with pytest.raises(ZeroDivisionError):
        optimizer.step(lambda: 1 / 0)
    optimizer.step()
    assert seen == [1, 2, 3]


def test_a_function_mode_sees_the_step_range():
    class Mode(TorchFunctionMode):
        def __init__(self):
            self.seen = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen.append(func.__name__)
            return func(*args, **(kwargs or {}))

    optimizer = _optimizer()
    with Mode() as mode:
        assert _group_walk.observed()
        optimizer.step()
    assert "_record_function_enter_new" in mode.seen and optimizer.updates == 1
    assert not _group_walk.observed()


@pytest.mark.parametrize("scope", ["optimizer", "global"])
def test_a_post_hook_registered_by_the_closure_runs_after_the_step(scope):
    optimizer, seen, handles = _optimizer(), [], []

    def hook(o, args, kwargs):
        seen.append((o.updates, len(args), tuple(kwargs)))

    def closure():
        handles.append(optimizer.register_step_post_hook(hook) if scope == "optimizer"
                       else register_optimizer_step_post_hook(hook))
        return 3.0

    try:
        assert optimizer.step(closure=closure) == 3.0
    finally:
        handles[0].remove()
    assert seen == [(1, 1, ("closure",))]


def test_an_unobserved_step_ends_in_the_step_code_method():
    class Traced(Counting):
        def _optimizer_step_code(self):
            self.updates += 10

    optimizer = _optimizer(Traced)
    optimizer.step()
    assert optimizer.updates == 11


def test_a_compiled_step_traces_torchs_wrapper():
    class Logging(Counting):
        def _step_group(self, group, formats, items, rng_step):
            log.append(torch.is_grad_enabled())

    log, optimizer = [], _optimizer(Logging)
    torch._dynamo.reset()
    compiled = torch.compile(optimizer.step, backend="eager")
    with warnings.catch_warnings(record=True) as caught:
        warnings.simplefilter("always")
        compiled()
        compiled()
    torch._dynamo.reset()
    assert log == [False, False]
    assert not [w for w in caught if "_group_walk" in str(w.message)]
