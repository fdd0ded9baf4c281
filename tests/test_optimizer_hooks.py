"""Step hooks and profiler ranges of MatrixOptimizer against those of a plain torch.optim.Optimizer: the same hooks, in the same
order, with the same arguments and results, whichever way a step takes."""

import copy
import pickle

import pytest
import torch
from torch.optim.optimizer import register_optimizer_step_post_hook, register_optimizer_step_pre_hook

from viola_amd.optim.matrix import MatrixOptimizer


class Ours(MatrixOptimizer):
    def __init__(self, params, log):
        super().__init__(params, dict(lr=.5))
        self.log = log

    def _step_local(self, parameter, gradient, state, group, index):
        self.log.append("update")
        parameter.sub_(gradient, alpha=group["lr"])


class Plain(torch.optim.Optimizer):
    def __init__(self, params, log):
        super().__init__(params, dict(lr=.5))
        self.log = log

    @torch.no_grad()
    def step(self, closure=None):
        loss = None
        if closure is not None:
            with torch.enable_grad():
                loss = closure()
        for group in self.param_groups:
            for p in group["params"]:
                if p.grad is not None:
                    self.log.append("update")
                    p.sub_(p.grad, alpha=group["lr"])
        return loss


def _made(cls):
    log, p = [], torch.nn.Parameter(torch.arange(6.).view(2, 3))
    p.grad = torch.ones_like(p)
    return cls([p], log), p, log


def _hook(log, name, result=None):
    def hook(optimizer, args, kwargs):
        log.append((name, len(args), args[0] is optimizer, sorted(kwargs)))
        return result(optimizer) if result else None
    return hook


def _compare(run):
    outcomes = []
    for cls in (Ours, Plain):
        optimizer, p, log = _made(cls)
        returned = run(optimizer, p, log)
        outcomes.append((log, p.detach().clone(), returned))
    (a, pa, ra), (b, pb, rb) = outcomes
    assert a == b and torch.equal(pa, pb) and ra == rb, (a, b, ra, rb)
    return a


def test_plain_steps():
    assert _compare(lambda o, p, log: o.step()) == ["update"]
    assert _compare(lambda o, p, log: o.step(lambda: 3.)) == ["update"]
    assert _compare(lambda o, p, log: o.step(closure=lambda: 3.)) == ["update"]


def test_hooks_run_in_order_and_can_be_removed():
    def run(o, p, log):
        handles = [o.register_step_pre_hook(_hook(log, "pre 1")), o.register_step_pre_hook(_hook(log, "pre 2")),
                   o.register_step_post_hook(_hook(log, "post 1")), o.register_step_post_hook(_hook(log, "post 2"))]
        o.step()
        for handle in handles:
            handle.remove()
        o.step()
    assert [entry[0] if isinstance(entry, tuple) else entry for entry in _compare(run)] == ["pre 1", "pre 2", "update", "post 1", "post 2", "update"]


def test_global_hooks_run_around_them():
    def run(o, p, log):
        handles = [register_optimizer_step_pre_hook(_hook(log, "global pre")), register_optimizer_step_post_hook(_hook(log, "global post"))]
        try:
            o.step()
            o.register_step_pre_hook(_hook(log, "pre"))
            o.register_step_post_hook(_hook(log, "post"))
            o.step()
        finally:
            for handle in handles:
                handle.remove()
        o.step()
    assert len(_compare(run)) == 12 - 1


def test_a_pre_hook_replaces_the_arguments():
    """A closure handed in by a hook is called, and post hooks see the new arguments."""
    def run(o, p, log):
        o.register_step_pre_hook(_hook(log, "pre", lambda optimizer: ((optimizer,), {"closure": lambda: log.append("closure") or 5.})))
        o.register_step_post_hook(_hook(log, "post"))
        return o.step()
    assert "closure" in _compare(run)


def test_a_pre_hook_with_a_wrong_result_raises():
    for cls in (Ours, Plain):
        optimizer, p, log = _made(cls)
        optimizer.register_step_pre_hook(lambda *_: 7)
        with pytest.raises(RuntimeError):
            optimizer.step()
        assert log == []


@pytest.mark.parametrize("others", [False, True])
def test_the_binding_runs_once_among_the_others(others):
    optimizer, p, log = _made(Ours)
    if others:
        optimizer.register_step_pre_hook(_hook(log, "pre"))
    optimizer.bind_step(_hook(log, "bind before"), _hook(log, "bind after"))
    if others:
        optimizer.register_step_post_hook(_hook(log, "post"))
    optimizer.step()
    names = [entry[0] if isinstance(entry, tuple) else entry for entry in log]
    assert names == (["pre"] if others else []) + ["bind before", "update", "bind after"] + (["post"] if others else [])
    assert all(entry[1:] == (1, True, []) for entry in log if isinstance(entry, tuple))


def test_profiler_ranges_are_there_while_one_runs():
    optimizer, p, _ = _made(Ours)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        optimizer.step()
        optimizer.zero_grad()
    names = [event.key for event in profile.key_averages()]
    assert "Optimizer.step#Ours.step" in names and "Optimizer.zero_grad#Ours.zero_grad" in names
    assert p.grad is None


def test_zero_grad_and_schedulers():
    optimizer, p, log = _made(Ours)
    optimizer.zero_grad(set_to_none=False)
    assert p.grad.count_nonzero() == 0
    optimizer.zero_grad()
    assert p.grad is None
    scheduler = torch.optim.lr_scheduler.StepLR(optimizer, 1, .5)
    p.grad = torch.ones_like(p)
    optimizer.step()
    scheduler.step()
    optimizer.step()
    assert log == ["update", "update"] and torch.allclose(p, torch.arange(6.).view(2, 3) - .75)


@pytest.mark.parametrize("how", [copy.deepcopy, lambda o: pickle.loads(pickle.dumps(o))])
def test_copies_step_as_torch_copies_do(how):
    """torch keeps the state, the groups and the defaults of a copied optimizer; its step runs all the same."""
    torch.manual_seed(0)
    p = torch.nn.Parameter(torch.ones(2, 3))
    copied = how(torch.optim.SGD([p], lr=.5)), how(_Stepper([p], dict(lr=.5)))
    for optimizer in copied:
        q = optimizer.param_groups[0]["params"][0]
        q.grad = torch.ones_like(q)
        if isinstance(optimizer, _Stepper):
            optimizer.skip_nonfinite = False                                       # a plain attribute, which no copy keeps
        optimizer.step()
        assert torch.equal(q.detach(), torch.full((2, 3), .5))


class _Stepper(MatrixOptimizer):
    def _step_local(self, parameter, gradient, state, group, index):
        parameter.sub_(gradient, alpha=group["lr"])
