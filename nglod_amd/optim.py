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
    shape, stride = p.shape, p.stride()
    for t in others:
        if t.shape != shape or t.stride() != stride:
            return False
    return True


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
            torch.autograd.graph.increment_version(list(params))
        return None

    def _plans(self):
        """[(group, params, grads, exp_avgs, exp_avg_sqs, step)], the states
        created and their steps counted; None where torch's step must run
        (and nothing has been touched)."""
        current = torch.cuda.current_device() if torch.cuda.is_available() else -1
        fresh = False
        found = []
        for group in self.param_groups:
            if (group["amsgrad"] or group["weight_decay"] != 0 or group["maximize"] or group["capturable"]
                    or group["differentiable"] or group.get("fused") or group["foreach"] is False
                    or isinstance(group["lr"], torch.Tensor)
                    or any(isinstance(b, torch.Tensor) for b in group["betas"])):
                return None
            rows = []
            for p in group["params"]:
                g = p.grad
                if g is None:
                    continue
                if (type(p) is not torch.nn.Parameter or not p.is_cuda or g.layout != torch.strided
                        or p.dtype != torch.float32 or g.dtype != torch.float32 or p.get_device() != current
                        or g.get_device() != current or not _dense_like(p, g)):
                    return None
                s = self.state.get(p)
                if not s:
                    fresh = True
                    continue
                avg, sq, step = s["exp_avg"], s["exp_avg_sq"], s["step"]
                if (avg.dtype != torch.float32 or sq.dtype != torch.float32 or avg.get_device() != current
                        or sq.get_device() != current or step.is_cuda or not _dense_like(p, avg, sq)):
                    return None
                rows.append((p, g, avg, sq, step))
            found.append((group, rows))
        if not fresh and not any(rows for _, rows in found):
            return None  # no gradients: nothing on any device
        if torch.cuda.is_current_stream_capturing():
            return None  # torch's step says what capture needs
        plans = []
        with torch.no_grad():
            for group, rows in found:
                if fresh:
                    params, grads, avgs, sqs, maxs, steps = [], [], [], [], [], []
                    self._init_group(group, params, grads, avgs, sqs, maxs, steps)
                    rows = list(zip(params, grads, avgs, sqs, steps))
                by_step = {}
                for row in rows:
                    by_step.setdefault(int(row[4].add_(1).item()), []).append(row[:4])
                for step, at in by_step.items():
                    plans.append((group, *zip(*at), step))
        return plans
