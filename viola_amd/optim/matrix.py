"""Base class for optimizers whose update needs a whole logical matrix
(viola/optim/matrix.py:14-135, plain-tensor path). One GPU: DTensor parameters, owner
gather/scatter and mesh all-reduces of the reference are not part of this build."""

import functools
from itertools import chain

import torch
from torch.autograd import profiler
from torch.optim.optimizer import _global_optimizer_post_hooks, _global_optimizer_pre_hooks


class MatrixOptimizer(torch.optim.Optimizer):
    """Subclasses implement `_step_local(parameter, gradient, state, group, index)` on full tensors;
    `index` is the parameter's stable position over all groups."""

    def __init__(self, params, defaults, *, shard_state=True, skip_nonfinite=False):
        self.shard_state = shard_state
        self.skip_nonfinite = skip_nonfinite
        self.step_was_skipped = False
        self._partition = None
        super().__init__(params, defaults)
        self.register_load_state_dict_pre_hook(self._before_load)
        self.register_load_state_dict_post_hook(self._after_load)

    @staticmethod
    def profile_hook_step(func):
        """The stock wrapper of `step` (hooks before and after, a profiler range around) without the range while no profiler
        runs: entering and leaving one costs about 6 us of host time, which a small model's step waits for."""
        recorded = torch.optim.Optimizer.profile_hook_step(func)

        @functools.wraps(func)
        def wrapper(self, *args, **kwargs):
            if profiler._is_profiler_enabled:
                return recorded(self, *args, **kwargs)
            args = (self, *args)
            for hook in chain(_global_optimizer_pre_hooks.values(), self._optimizer_step_pre_hooks.values()):
                result = hook(self, args, kwargs)
                if result is not None:
                    if not (isinstance(result, tuple) and len(result) == 2):
                        raise RuntimeError(f"{func} must return None or a tuple of (new_args, new_kwargs), but got {result}.")
                    args, kwargs = result
            out = func(*args, **kwargs)
            self._optimizer_step_code()
            for hook in chain(self._optimizer_step_post_hooks.values(), _global_optimizer_post_hooks.values()):
                hook(self, args, kwargs)
            return out

        return wrapper

    def zero_grad(self, set_to_none=True):
        if not set_to_none or profiler._is_profiler_enabled:
            return super().zero_grad(set_to_none)
        for group in self.param_groups:
            for param in group["params"]:
                if param.grad is not None:
                    param.grad = None

    def _step_local(self, parameter, gradient, state, group, index):
        raise NotImplementedError

    def _has_nonfinite(self):
        return any(not torch.isfinite(p.grad).all() for g in self.param_groups for p in g["params"] if p.grad is not None)

    @torch.no_grad()
    def step(self, closure=None):
        self.step_was_skipped = False
        loss = None
        if closure is not None:
            with torch.enable_grad():
                loss = closure()
        if self.skip_nonfinite and self._has_nonfinite():
            self.step_was_skipped = True
            return loss
        index = 0
        work = []
        for group in self.param_groups:
            stable = group.get("viola_parameter_indices")
            for local, param in enumerate(group["params"]):
                position = stable[local] if stable is not None else index
                index += 1
                if param.grad is None:          # no decay, no state advance for a missing gradient
                    continue
                work.append((param, param.grad, self.state[param], group, position))
        self._step_all(work)
        return loss

    def _step_all(self, work):
        """All (parameter, gradient, state, group, index) of one step; subclasses may batch equal shapes."""
        for item in work:
            self._step_local(*item)

    # Optimizer.load_state_dict casts floating state tensors to the parameter's dtype, which would
    # destroy the raw uint8 FP8 payload / fp32 scales / bf16 moments. Tensors are therefore set
    # aside before the stock loader runs and put back verbatim afterwards.
    def _before_load(self, optimizer, saved):
        saved = dict(saved)
        is_tensor = lambda v: isinstance(v, torch.Tensor)
        self._held = {pid: {k: v for k, v in state.items() if is_tensor(v)} for pid, state in saved["state"].items()}
        self._held_groups = saved["param_groups"]
        saved["state"] = {pid: {k: v for k, v in state.items() if not is_tensor(v)} for pid, state in saved["state"].items()}
        return saved

    def _after_load(self, optimizer):
        for old, group in zip(self._held_groups, self.param_groups):
            for pid, param in zip(old["params"], group["params"]):
                for name, value in self._held.get(pid, {}).items():
                    self.state[param][name] = value.to(device=param.device)
        del self._held, self._held_groups
