"""SparseGaussianAdam: same class and behaviour as the reference's `fast_2d_gs/sparse_gaussian_adam.py` (lines 10-49),
driving the HIP masked-Adam kernel through the operator boundary."""
import torch
import torch.optim

from fast_sp_gs_amd._C import get_C_function
from fast_sp_gs_amd.lib import host

__all__ = ['SparseGaussianAdam', 'DenseAdam']


class SparseGaussianAdam(torch.optim.Adam):
    _update_C = staticmethod(get_C_function('AdamMasksedUpdated'))

    def __init__(self, params, lr, eps):
        super().__init__(params=params, lr=lr, eps=eps)
        self.N = None
        self.visibility = None

    def _state_of(self, param):
        """The parameter's optimiser state; created on first use with the keys torch's Adam uses
        (sparse_gaussian_adam.py:28-33), so checkpoints of either optimiser load into the other."""
        state = self.state[param]
        if not state:
            state.update(step=torch.zeros((), dtype=torch.float32),
                         exp_avg=torch.zeros_like(param, memory_format=torch.preserve_format),
                         exp_avg_sq=torch.zeros_like(param, memory_format=torch.preserve_format))
        return state

    @torch.no_grad()
    def step(self):
        """One masked Adam update of every parameter group that has a gradient (sparse_gaussian_adam.py:20-45), the
        groups' kernels folded into one launch; the arithmetic per element is the single-tensor
        kernel's. The call advances the step counts and forms the bias corrections as well."""
        jobs = []  # (param, grad, first moment, second moment, step count, rate, eps)
        for group in self.param_groups:
            if len(group["params"]) != 1:
                raise AssertionError("more than one tensor in group")
            param = group["params"][0]
            if param.grad is None or param.grad.numel() == 0:
                continue
            state = self._state_of(param)
            jobs.append((param, param.grad, state["exp_avg"], state["exp_avg_sq"], state["step"], group["lr"], group["eps"]))
        if jobs:
            p, g, m, v, steps, rates, epss = map(list, zip(*jobs))
            host.adam_masked_step(p, g, m, v, steps, self.visibility, rates, 0.9, 0.999, epss, self.N)

    def set_before_step(self, visibility, N):
        self.visibility, self.N = visibility, N


class DenseAdam(torch.optim.Adam):
    """torch.optim.Adam with the plain update (no weight decay, amsgrad, maximize, capturable) of all of a group's float32
    tensors in one launch; state keys as torch's, so checkpoints load either way. Any other setting takes torch's step. As
    with torch's fused step the parameters' version counters stay: whoever keeps copies of them (`DeformNetwork.pack`)
    refreshes those itself."""

    def __setstate__(self, state):
        super().__setstate__(state)
        # one step count per parameter, also where the loaded state shares tensors (between parameters, or with the optimiser
        # it was taken from): torch's step advances each parameter's in place
        for entry in self.state.values():
            if isinstance(entry.get('step'), torch.Tensor):
                entry['step'] = entry['step'].clone()

    @torch.no_grad()
    def step(self, closure=None):
        groups = self.param_groups
        if closure is not None or any(g['weight_decay'] or g['amsgrad'] or g['maximize'] or g['capturable'] or g['fused'] or
                                      g['differentiable'] or isinstance(g['lr'], torch.Tensor) for g in groups):
            return super().step(closure)
        if any(p.grad is not None and (p.grad.is_sparse or p.dtype != torch.float32 or not p.is_cuda or not p.is_contiguous())
               for g in groups for p in g['params']):
            return super().step()
        for group in groups:
            params = [p for p in group['params'] if p.grad is not None]
            if not params:
                continue
            for p in params:
                if not self.state[p]:
                    self.state[p].update(step=torch.zeros((), dtype=torch.float32), exp_avg=torch.zeros_like(p),
                                         exp_avg_sq=torch.zeros_like(p))
            states = [self.state[p] for p in params]
            # the call advances the step counts too: 27 additions to host tensors through torch are 100 us
            host.adam_dense(params, [p.grad for p in params], [s['exp_avg'] for s in states],
                            [s['exp_avg_sq'] for s in states], [s['step'] for s in states], group['lr'], *group['betas'],
                            group['eps'])
