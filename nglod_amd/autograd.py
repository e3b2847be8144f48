"""torch.autograd.Function around the fused HIP query (OctreeSDF.sdf) with the
hand-written backward: parameter gradients by nglod_sdf_bwd, computed
deterministically (no float atomics), and position gradients (when the query
points require grad) by nglod_sdf_grad, the derivative torch autograd takes
through grid_sample, the decoder and ReLU.  First order only: the backward
itself is not differentiable (gradient penalties through it raise)."""
import torch
from torch.autograd.function import once_differentiable

from . import _lib


def _param_slots(net, params):
    """(kind, index) of each parameter; (None, -1) for one outside the grids and
    decoders.  Found by identity; one that is not read as it is (a grid's under a
    parametrization or a pruning mask) by its name, as its level's grid.  A decoder's
    raises: the gradient is that of the weight it is turned into."""
    slots = {}
    for i, f in enumerate(net.features):
        slots.setdefault(id(f.fm), ("grid", i))
    for i, l in enumerate(net.louts):
        first, _, last, *_ = l
        slots.setdefault(id(first.weight), ("w0", i))
        slots.setdefault(id(first.bias), ("b0", i))
        slots.setdefault(id(last.weight), ("w1", i))
        slots.setdefault(id(last.bias), ("b1", i))
    found = [slots.get(id(p)) for p in params]
    if None in found:
        names = {id(p): name for name, p in net.named_parameters()}
        found = [s if s is not None else _slot_of(names[id(p)]) for s, p in zip(found, params)]
    return found


def _slot_of(name):
    parts = name.split(".")
    if parts[0] == "features":
        return "grid", int(parts[1])
    if parts[0] == "louts":
        raise KeyError(f"no gradient for {name}: not a weight or bias of its decoder")
    return None, -1


# A forward of every level whose caller runs the backward itself, with nothing in
# between, keeps its features for it (164 bytes per query and level) up to this many
# bytes; a larger batch computes them again, and so does any other backward: a
# program may write the weights in between, and a write through .data leaves no mark
# to know it by.
SAVE_LIMIT = 4 << 30


def _versions(params):
    return [(p.data_ptr(), p._version) for p in params]


class _SdfFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, net, x, lod, all_levels, keep_features, *params):
        ctx.net = net
        ctx.lod = lod
        ctx.all_levels = all_levels
        xf = x.detach().reshape(-1, 3).float().contiguous()
        ctx.x_shape = x.shape
        ctx.x_dtype = x.dtype
        n = xf.shape[0]
        if keep_features and all_levels and n > 0 and any(ctx.needs_input_grad[5:]):
            lib = _lib.load()
            m = net.descriptor(_lib.FP32)
            nbytes = lib.nglod_sdf_fwd_save_bytes(m, n, lod)
            if nbytes <= SAVE_LIMIT and n <= 1 << 28:
                out = torch.empty(lod + 1, n, 1, device=x.device, dtype=torch.float32)
                saved = torch.empty(nbytes, device=x.device, dtype=torch.uint8)
                ws = torch.empty(lib.nglod_sdf_fwd_save_workspace_size(n), device=x.device, dtype=torch.uint8)
                _lib.check(lib.nglod_sdf_fwd_save(m, _lib.ptr(xf), n, lod, _lib.ptr(out), _lib.ptr(saved), nbytes,
                                                  _lib.ptr(ws), ws.numel(), _lib.stream_of(x)), "nglod_sdf_fwd_save")
                ctx.versions = _versions(params)
                ctx.save_for_backward(xf, saved)
                return out
        ctx.save_for_backward(xf)
        if all_levels:
            return torch.stack(net.sdf_all_hip(xf, lod), 0)
        return net.sdf_hip(xf, lod)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_out):
        x, *saved = ctx.saved_tensors
        net, L = ctx.net, ctx.lod
        n = x.shape[0]
        dev = x.device
        if ctx.all_levels:
            g = grad_out[..., 0].float().contiguous()  # [L+1, n]
            mask = (1 << (L + 1)) - 1
        else:
            g = torch.zeros(L + 1, n, dtype=torch.float32, device=dev)
            g[L] = grad_out[:, 0].float()
            mask = 1 << L
        grad_x = None
        if ctx.needs_input_grad[1]:
            # sum over the decoded levels of d loss / d d_l * d d_l / d x
            grad_x = torch.zeros(n, 3, dtype=torch.float32, device=dev)
            for lvl in range(L + 1):
                if (mask >> lvl) & 1:
                    grad_x.addcmul_(g[lvl][:, None], net.sdf_grad_hip(x, lvl)[1])
            grad_x = grad_x.to(ctx.x_dtype).reshape(ctx.x_shape)
        if not any(ctx.needs_input_grad[5:]):
            return (None, grad_x, None, None, None, *([None] * len(ctx.needs_input_grad[5:])))
        used_dec = {0} if net.num_decoder == 1 else {i for i in range(L + 1) if (mask >> i) & 1}
        G = _lib.NglodModelGrads()
        out = {}
        for i, f in enumerate(net.features):
            if i <= L:
                t = torch.empty_like(f.fm, memory_format=torch.channels_last_3d)
                out[("grid", i)] = t
                G.grid[i] = t.data_ptr()
        for d, l in enumerate(net.louts):
            for key, p in (("w0", l[0].weight), ("b0", l[0].bias), ("w1", l[2].weight), ("b1", l[2].bias)):
                t = torch.empty_like(p, memory_format=torch.contiguous_format)
                out[(key, d)] = t
                getattr(G, key)[d] = t.data_ptr()
        m = net.descriptor(_lib.FP32)
        lib = _lib.load()
        params = _lib.parameter_list(net)
        # features of other weights are not the features of these: computed again
        if saved and ctx.versions == _versions(params):
            nbytes = lib.nglod_sdf_bwd_saved_workspace_size(m, n, L)
            ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device=dev)
            _lib.check(lib.nglod_sdf_bwd_saved(m, _lib.ptr(x), n, L, _lib.ptr(g), mask, G, _lib.ptr(saved[0]),
                                               saved[0].numel(), _lib.ptr(ws), ws.numel(), _lib.stream_of(x)),
                       "nglod_sdf_bwd_saved")
        else:
            nbytes = lib.nglod_sdf_bwd_workspace_size(m, n, L)
            ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device=dev)
            _lib.check(lib.nglod_sdf_bwd(m, _lib.ptr(x), n, L, _lib.ptr(g), mask, G, _lib.ptr(ws), ws.numel(),
                                         _lib.stream_of(x)), "nglod_sdf_bwd")
        grads = []
        for kind, idx in _param_slots(net, params):
            if kind == "grid":
                grads.append(out.get(("grid", idx)))
            elif kind is not None and idx in used_dec:
                grads.append(out[(kind, idx)])
            else:
                grads.append(None)
        return (None, grad_x, None, None, None, *grads)


def sdf_with_grad(net, x, lod, all_levels, stacked=False, params=None, keep_features=False):
    """stacked: the levels' predictions as one [lod + 1, n, 1] tensor; params:
    net's parameters, if the caller has them; keep_features: the caller runs the
    backward before anything can write the weights."""
    if params is None:
        params = _lib.parameter_list(net)
    out = _SdfFunction.apply(net, x, lod, all_levels, keep_features, *params)
    if all_levels and not stacked:
        return [out[i] for i in range(out.shape[0])]
    return out
