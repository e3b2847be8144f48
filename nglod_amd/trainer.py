"""Training step of the dense model (Trainer.step_geometry,
sdf-net/lib/trainer.py:294-340) on the HIP path, and the seeded fit that
produces the benchmark model.

step_geometry: zero_grad; predictions of every LOD in loss_lods from one
fused forward (the reference's return_lst branch, :317-319); loss =
sum over LODs of sum (pred - gt)^2, divided by the batch size (:325-337), and
its gradient from one kernel (nglod_geometry_loss); backward through
nglod_sdf_bwd_saved; Adam (lr 1e-3, :184-185) by nglod_adam_step.
"""
import torch

from . import _lib, workloads
from .autograd import sdf_with_grad
from .meshdata import MeshData
from .octree_sdf import OctreeSDF
from .optim import Adam
from . import mesh as _mesh


def _training(module):
    """Whether module and everything in it is in training mode."""
    return module.training and all(_training(m) for m in module._modules.values() if m is not None)


class Trainer:
    def __init__(self, net, lr=1e-3, loss_lods=None):
        self.net = net
        self.optimizer = Adam(net.parameters(), lr=lr)
        self.loss_lods = list(range(net.num_lods)) if loss_lods is None else list(loss_lods)
        self.last_loss = None

    def _fused(self, pts, gts, params):
        """Whether loss and gradient can come from nglod_geometry_loss: a plain
        OctreeSDF's every-level predictions against one FP32 value per point."""
        net = self.net
        return (type(net) is OctreeSDF and "sdf" not in net.__dict__ and net.lod is None and pts.dim() == 2
                and pts.is_cuda and pts.shape[0] > 0 and torch.is_tensor(gts) and gts.shape == (pts.shape[0], 1)
                and gts.dtype == torch.float32 and gts.device == pts.device and not gts.requires_grad
                and torch.is_grad_enabled()
                and all(0 <= i < net.num_lods for i in self.loss_lods)
                and len(set(self.loss_lods)) == len(self.loss_lods) > 0
                and all(p.requires_grad for p in params))

    def step_geometry(self, pts, gts):
        net = self.net
        params = _lib.parameter_list(net)
        if type(net) is not OctreeSDF:
            net.train()
            net.zero_grad()
        else:
            if not _training(net):
                net.train()
            for p in params:
                p.grad = None
        batch_size = pts.shape[0]
        if self._fused(pts, gts, params):
            stacked = sdf_with_grad(net, pts, net.num_lods - 1, all_levels=True, stacked=True, params=params,
                                    keep_features=True)
            net.loss_preds = list(stacked.unbind(0))
            gt = gts.contiguous()
            grad = torch.empty_like(stacked)
            loss = torch.empty((), dtype=torch.float32, device=pts.device)
            lib = _lib.load()
            ws = torch.empty(lib.nglod_geometry_loss_workspace_size(), dtype=torch.uint8, device=pts.device)
            _lib.check(lib.nglod_geometry_loss(_lib.ptr(stacked), _lib.ptr(gt), batch_size, net.num_lods,
                                               sum(1 << i for i in self.loss_lods), _lib.ptr(grad), _lib.ptr(loss),
                                               _lib.ptr(ws), ws.numel(), _lib.stream_of(pts)), "nglod_geometry_loss")
            torch.autograd.backward(stacked, grad)
            self.optimizer.step()
            self.last_loss = loss
            return self.last_loss
        preds = net.sdf(pts, return_lst=True)
        preds = [preds[i] for i in self.loss_lods]
        loss = 0.0
        for pred in preds:
            loss = loss + ((pred - gts) ** 2).sum()
        loss = loss / batch_size
        loss.backward()
        self.optimizer.step()
        self.last_loss = loss.detach()
        return self.last_loss


def fit(net, md, iterations=200, batch=2 ** 17, seed=0, lr=1e-3):
    """Seeded fit of `net` to the mesh held by `md` (MeshData)."""
    tr = Trainer(net, lr=lr)
    for it in range(iterations):
        pts, gts = md.training_batch(batch, seed=seed * 100003 + it)
        tr.step_geometry(pts, gts)
    return tr


def fitted_icosphere_model(seed=0, device="cuda", iterations=200, batch=2 ** 17, lr=1e-3, pos_invariant=True):
    """The benchmark model: 5-LOD OctreeSDF (seeded init) fitted for
    `iterations` Adam steps to the seeded displaced level-4 icosphere."""
    net = workloads.make_model(num_lods=5, pos_invariant=pos_invariant, seed=seed, device=device)
    V, F = _mesh.displaced_icosphere(seed)
    md = MeshData(V, F, device)
    fit(net, md, iterations=iterations, batch=batch, seed=seed, lr=lr)
    net.eval()
    return net, md
