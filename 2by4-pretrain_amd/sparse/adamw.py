"""AdamW with the masked decay of the 2:4 recipe folded into the update (one HIP launch for all
tensors of a parameter group).

The reference trains with its AdamW (sparse/adamw.py:9-115) after a loop that adds the decay term
to the gradients of masked weights (README.md:205-213):

    p.grad = p.grad.float(); masked_add_(p.grad.data, p.data, p.mask, alpha=alpha); p.cnt = 0

MaskedDecayAdamW does both in one pass per parameter: for a parameter that carries a `mask` and is
in 'sparse' mode the gradient seen by the update is grad + alpha * p where the mask is zero, then
the update of sparse/adamw.py:70-113 (decoupled weight decay, bias-corrected moments, no amsgrad).
The stored gradient is not modified; `cnt` is reset as the loop above does.  Parameters and moments
are float32; gradients may be float32, float16 or bfloat16.

capturable=True keeps every parameter's step count in device memory (an int64 tensor, advanced by a
device operation), as torch's own optimizers do under that name: a step recorded into a HIP graph then
replays with the count of the replay.  Hyper-parameters are read on the host at every call, so a
recording holds the values of its time.
"""
import struct

import torch
from torch.optim.optimizer import Optimizer

from . import _native as N

__all__ = ["MaskedDecayAdamW"]


def _rounds(params):
    """`params` as lists in which no memory stands twice: the tensors of one launch are updated side by side, and those
    that overlap (a parameter listed twice, of which torch warns, or views of one buffer) one after the other, in the
    order of the list."""
    spans = [(p.data_ptr(), p.numel() * p.element_size()) for p in params]
    in_memory = sorted(span for span in spans if span[1])
    if all(start + size <= after for (start, size), (after, _) in zip(in_memory, in_memory[1:])):
        return [params]
    rounds, turns = [], []
    for p, (start, size) in zip(params, spans):
        turns.append(1 + max((turn for turn, (other, extent) in zip(turns, spans) if other < start + size and start < other + extent), default=-1))
        if turns[-1] == len(rounds):
            rounds.append([])
        rounds[turns[-1]].append(p)
    return rounds


class MaskedDecayAdamW(Optimizer):
    def __init__(self, params, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=1e-2, alpha=0.0, capturable=False):
        if not 0.0 <= lr:
            raise ValueError("Invalid learning rate: {}".format(lr))
        if not 0.0 <= eps:
            raise ValueError("Invalid epsilon value: {}".format(eps))
        if not 0.0 <= betas[0] < 1.0:
            raise ValueError("Invalid beta parameter at index 0: {}".format(betas[0]))
        if not 0.0 <= betas[1] < 1.0:
            raise ValueError("Invalid beta parameter at index 1: {}".format(betas[1]))
        super().__init__(params, dict(lr=lr, betas=betas, eps=eps, weight_decay=weight_decay, alpha=alpha,
                                      capturable=bool(capturable)))

    def __setstate__(self, state):
        super().__setstate__(state)
        for of_p in self.state.values():         # (load_state_dict makes float32 of a capturable optimizer's step counts)
            if torch.is_tensor(of_p.get("step")):
                of_p["step"] = of_p["step"].to(torch.int64)

    def _check(self, p, capturable=False):
        """Once per parameter: what the kernel assumes about it (flat float32 storage shared by the moments)."""
        if p.dtype != torch.float32 or not p.is_cuda:
            raise RuntimeError("MaskedDecayAdamW: parameters must be float32 GPU tensors")
        if not (p.is_contiguous() or (p.dim() == 2 and p.t().is_contiguous())):
            raise RuntimeError("MaskedDecayAdamW: parameters must be dense in memory")
        return {"step": torch.zeros((), dtype=torch.int64, device=p.device) if capturable else 0,
                "exp_avg": torch.empty_like(p, memory_format=torch.preserve_format),       # zeroed with the others of the
                "exp_avg_sq": torch.empty_like(p, memory_format=torch.preserve_format)}    # group, in one launch (step)

    @torch.no_grad()
    def step(self, closure=None):
        loss = None
        if closure is not None:
            with torch.enable_grad():
                loss = closure()
        for group, params in ((group, params) for group in self.param_groups for params in _rounds(group["params"])):
            beta1, beta2 = group["betas"]
            lr, eps, wd, alpha = float(group["lr"]), float(group["eps"]), float(group["weight_decay"]), float(group["alpha"])
            # Everything is looked at before anything is launched; the tensors of one launch share the types of
            # gradient and mask and a host-side step count (device-side counts travel with their tensor)
            entries, counts, launches, fresh, negated, codes = [], [], {}, [], [], N.dtype_codes
            for p in params:
                grad = p.grad
                if grad is None:
                    continue
                state = self.state[p]
                if not state:
                    state = self._check(p, group.get("capturable", False))
                    fresh.append((p, state))                       # the optimizer's own only once it holds zeros
                stride = p.stride()
                if grad.is_sparse or grad.stride() != stride:
                    raise RuntimeError("MaskedDecayAdamW: the gradient must be dense with the parameter's strides")
                mask = getattr(p, "mask", None)
                if mask is not None and not (torch.is_tensor(mask) and getattr(p, "mode", "sparse") == "sparse"):
                    mask = None
                if mask is not None and (mask.stride() != stride or mask.device != p.device):
                    raise RuntimeError("MaskedDecayAdamW: mask must have the parameter's strides and device")
                if grad.is_neg():                                  # (the kernel reads and writes storage)
                    grad = grad.resolve_neg()
                step = state["step"]
                on_device = type(step) is not int and torch.is_tensor(step)
                if on_device:
                    counts.append(step)
                entries.append((p, grad, state, mask, codes[grad.dtype], N.U8 if mask is None else codes[mask.dtype], on_device))
            if fresh:
                torch._foreach_zero_([state[name] for _, state in fresh for name in ("exp_avg", "exp_avg_sq")])
                for p, state in fresh:
                    self.state[p] = state
            if counts:
                torch._foreach_add_(counts, 1)
            for p, grad, state, mask, grad_code, mask_code, on_device in entries:
                if on_device:
                    key, step_ptr = (grad_code, mask_code, 0), state["step"].data_ptr()
                else:
                    step = state["step"] = state["step"] + 1
                    key, step_ptr = (grad_code, mask_code, step), 0
                if mask is not None:
                    p.cnt = 0
                values = p
                if p.is_neg():                                     # (updated beside, and written back through the view)
                    values = p.resolve_neg()
                    negated.append((p, values))
                launches.setdefault(key, []).extend((values.data_ptr(), grad.data_ptr(), state["exp_avg"].data_ptr(), state["exp_avg_sq"].data_ptr(),
                                                     0 if mask is None else mask.data_ptr(), step_ptr, p.numel()))
            for (grad_code, mask_code, step), words in launches.items():
                N.check(N.lib().tf24_adamw_masked_decay_list(struct.pack("%dq" % len(words), *words), len(words) // 7, grad_code, mask_code,
                                                             lr, float(beta1), float(beta2), eps, wd, alpha, step, N.stream_ptr()))
            for p, values in negated:
                p.copy_(values)
        return loss
