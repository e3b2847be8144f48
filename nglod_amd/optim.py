"""torch.optim.Adam with its update in one HIP launch.

Same class, arguments, state and results (bit for bit: nglod_adam_step rounds
as torch's multi-tensor update on this GPU); the plain FP32 case on the GPU
runs nglod_adam_step, anything else torch's own step.
"""
import ctypes

import torch

from . import _lib


def _dense_like(p, *others):
    """Whether p is laid out without gaps and the others exactly as p."""
    if not (p.is_contiguous() or (p.dim() == 5 and p.is_contiguous(memory_format=torch.channels_last_3d))):
        return False
    return all(t.stride() == p.stride() and t.shape == p.shape for t in others)


class Adam(torch.optim.Adam):
    def step(self, closure=None):
        plans = None if closure is not None or torch.is_grad_enabled() and self.defaults.get("differentiable") \
            else self._plans()
        if plans is None:
            base = torch.optim.Adam.step
            # a hooked base step would run this class's step hooks a second time
            return (base.__wrapped__ if getattr(base, "hooked", False) else base)(self, closure)
        lib = _lib.load()
        for group, params, grads, avgs, sqs, step in plans:
            k = len(params)
            arr = ctypes.c_void_p * k
            beta1, beta2 = group["betas"]
            _lib.check(lib.nglod_adam_step(arr(*[p.data_ptr() for p in params]), arr(*[g.data_ptr() for g in grads]),
                                           arr(*[m.data_ptr() for m in avgs]), arr(*[v.data_ptr() for v in sqs]),
                                           (ctypes.c_int64 * k)(*[p.numel() for p in params]), k, float(beta1),
                                           float(beta2), float(group["eps"]), float(group["lr"]), step,
                                           _lib.stream_of(params[0])), "nglod_adam_step")
            # written behind autograd's back: what is keyed by a version must see it
            torch.autograd.graph.increment_version(params)
        return None

    def _plans(self):
        """[(group, params, grads, exp_avgs, exp_avg_sqs, step)], the states
        created and their steps counted; None where torch's step must run
        (and nothing has been touched)."""
        for group in self.param_groups:
            if (group["amsgrad"] or group["weight_decay"] != 0 or group["maximize"] or group["capturable"]
                    or group["differentiable"] or group.get("fused") or group["foreach"] is False
                    or isinstance(group["lr"], torch.Tensor)
                    or any(isinstance(b, torch.Tensor) for b in group["betas"])):
                return None
            for p in group["params"]:
                g = p.grad
                if g is None:
                    continue
                if (g.is_sparse or p.dtype != torch.float32 or g.dtype != torch.float32 or not p.is_cuda
                        or type(p) is not torch.nn.Parameter or p.device != g.device
                        or p.device.index != torch.cuda.current_device() or not _dense_like(p, g)):
                    return None
                s = self.state.get(p)
                if s and (not _dense_like(p, s["exp_avg"], s["exp_avg_sq"]) or s["step"].is_cuda
                          or s["exp_avg"].dtype != torch.float32 or s["exp_avg_sq"].dtype != torch.float32
                          or s["exp_avg"].device != p.device or s["exp_avg_sq"].device != p.device):
                    return None
        if torch.cuda.is_current_stream_capturing():
            return None  # torch's step says what capture needs
        plans = []
        with torch.no_grad():
            for group in self.param_groups:
                params, grads, avgs, sqs, maxs, steps = [], [], [], [], [], []
                self._init_group(group, params, grads, avgs, sqs, maxs, steps)
                if not params:
                    continue
                torch._foreach_add_(steps, 1)
                by_step = {}
                for i, t in enumerate(steps):
                    by_step.setdefault(int(t.item()), []).append(i)
                for step, at in by_step.items():
                    pick = lambda v: [v[i] for i in at]
                    plans.append((group, pick(params), pick(grads), pick(avgs), pick(sqs), step))
        return plans
