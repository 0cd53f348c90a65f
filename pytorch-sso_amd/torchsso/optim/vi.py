"""VIOptimizer: Noisy K-FAC / variational inference on top of SecondOrderOptimizer.

Constructor arguments, `param_groups` / `defaults` keys and the `step` /
`prediction` contract are those of torchsso/optim/vi.py:11-299 of the reference.
The posterior of a layer is Gaussian with the mean kept in group['mean'] and the
covariance std_scale^2 * (A^-1 (x) G^-1).  A step draws `num_mc_samples` weight
samples (one batched call into the HIP engine for all layers; the noise comes
from torch's generator, one [dG, dA] matrix per Kronecker layer in param_group
order after manual_seed(step + seed), which is the order in which the reference
consumes it), averages gradients and curvature factors over the samples, and
runs the phases of SecondOrderOptimizer on the means.

The KL bookkeeping is a pure function here (`kl_rate`): the weight of the KL
term at step s relative to the initial one, from which the l2 coefficient and
the posterior scale of every group follow.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from torchsso.curv import curvature as _curv
from torchsso.optim.secondorder import SecondOrderOptimizer


def kl_rate(step, warmup_steps, init_kl, target_kl):
    """KL weight after `step` updates divided by the initial KL weight.

    Without warm-up the weight never moves.  With it, the weight goes linearly from
    `init_kl` to `target_kl` over `warmup_steps` updates and then stays
    (reference: vi.py:150-172, which returns without touching anything once
    step > warmup_steps: the value of the last whole step inside the warm-up holds)."""
    if warmup_steps is None:
        return 1.
    s = min(step, math.floor(warmup_steps))
    if s <= 0:
        return 1.
    return (init_kl + s / warmup_steps * (target_kl - init_kl)) / init_kl


def class_probabilities(output):
    """softmax over classes for [n, classes] logits, sigmoid for a vector of n logits."""
    output = output.detach()
    if output.ndim == 2:
        return F.softmax(output, dim=1)
    if output.ndim == 1:
        return torch.sigmoid(output)
    raise ValueError(f'Invalid ndim {output.ndim}')


def _running_sum(total, value, weight):
    return value * weight if total is None else torch.add(total, value, alpha=weight)


class VIOptimizer(SecondOrderOptimizer):
    r"""Variational-inference optimizer (arguments as the reference,
    vi.py:17-48): `dataset_size` scales the KL term, `num_mc_samples` /
    `val_num_mc_samples` are the numbers of posterior samples for training /
    prediction, `kl_weighting` (optionally warmed up from
    `warmup_kl_weighting_init` over `warmup_kl_weighting_steps`),
    `prior_variance`, `init_precision`, `seed`, `total_steps`."""

    _fuse_running_average = False    # the MC loop accumulates the raw factors

    def __init__(self, model: nn.Module, dataset_size: float, curv_type: str, curv_shapes: dict,
                 curv_kwargs: dict,
                 lr=0.01, momentum=0., momentum_type='preconditioned',
                 grad_ema_decay=1., grad_ema_type='raw', weight_decay=0.,
                 normalizing_weights=False, weight_scale=None,
                 acc_steps=1, non_reg_for_bn=False, bias_correction=False,
                 lars=False, lars_type='preconditioned',
                 num_mc_samples=10, val_num_mc_samples=10,
                 kl_weighting=1, warmup_kl_weighting_init=0.01, warmup_kl_weighting_steps=None,
                 prior_variance=1, init_precision=None,
                 seed=1, total_steps=1000):
        warm = warmup_kl_weighting_steps is not None
        for broken, what, value in (
                (dataset_size < 0, 'dataset size', dataset_size),
                (num_mc_samples < 1, 'number of MC samples', num_mc_samples),
                (val_num_mc_samples < 0, 'number of MC samples for validation', val_num_mc_samples),
                (kl_weighting < 0, 'KL weighting', kl_weighting),
                (warm and warmup_kl_weighting_init < 0, 'initial KL weighting',
                 warmup_kl_weighting_init),
                (prior_variance < 0, 'prior variance', prior_variance),
                (init_precision is not None and init_precision < 0, 'initial precision',
                 init_precision)):
            if broken:
                raise ValueError('Invalid {}: {}'.format(what, value))

        # KL weight the run starts with; the l2 coefficient is the gradient of the prior
        # term (0 switches the prior, and with it the sampling, off)
        kl0 = warmup_kl_weighting_init if warm else kl_weighting
        prior_l2 = 0 if prior_variance == 0 else kl0 / dataset_size / prior_variance
        posterior_scale = math.sqrt(kl0 / dataset_size)

        super(VIOptimizer, self).__init__(
            model, curv_type, curv_shapes, curv_kwargs, lr=lr, momentum=momentum,
            momentum_type=momentum_type, grad_ema_decay=grad_ema_decay,
            grad_ema_type=grad_ema_type, l2_reg=prior_l2, weight_decay=weight_decay,
            normalizing_weights=normalizing_weights, weight_scale=weight_scale,
            acc_steps=acc_steps, non_reg_for_bn=non_reg_for_bn, bias_correction=bias_correction,
            lars=lars, lars_type=lars_type)

        self.defaults.update(
            std_scale=posterior_scale, kl_weighting=kl_weighting,
            warmup_kl_weighting_init=warmup_kl_weighting_init,
            warmup_kl_weighting_steps=warmup_kl_weighting_steps,
            num_mc_samples=num_mc_samples, val_num_mc_samples=val_num_mc_samples,
            total_steps=total_steps, seed_base=seed)

        for group in self.param_groups:
            # a group without prior term (BatchNorm under non_reg_for_bn, or prior_variance
            # 0) is not sampled either
            group['std_scale'] = posterior_scale if group['l2_reg'] != 0 else 0
            group['mean'] = [p.data.detach().clone() for p in group['params']]
            self.init_buffer(group['mean'])

        if init_precision is not None:
            # a posterior to sample from before the first update: precision * I per layer
            curvs = [group['curv'] for group in self.param_groups]
            for curv in curvs:
                curv.element_wise_init(init_precision)
            _curv.step_all(curvs, update_std=self._sampled(self.param_groups))

    @staticmethod
    def _sampled(groups):
        return [group['std_scale'] > 0 for group in groups]

    # ---- gradients, seeds ----------------------------------------------------------

    def zero_grad(self, set_to_none=False):
        """Clears the gradients of the parameters and of the posterior means."""
        dense = []
        for group in self.param_groups:
            for t in list(group['mean']) + list(group['params']):
                if t.grad is not None:
                    t.grad.detach_()
                    if t.grad.layout == torch.strided:
                        dense.append(t.grad)
                    else:
                        t.grad.zero_()
        if dense:
            torch._foreach_zero_(dense)          # (one launch instead of one per tensor)

    @property
    def seed(self):
        return self.optim_state['step'] + self.defaults['seed_base']

    def set_random_seed(self, seed=None):
        seed = self.seed if seed is None else seed
        torch.manual_seed(seed)
        if torch.cuda.is_available():
            torch.cuda.manual_seed_all(seed)

    # ---- posterior <-> parameters --------------------------------------------------

    def sample_params(self):
        """Params <- a sample from the posterior where a std exists, else the mean
        (reference: vi.py:129-139)."""
        drawn, plain = [], []
        for group in self.param_groups:
            curv = group['curv']
            if curv is not None and curv.std is not None:
                drawn.append((curv, group['params'], group['mean'], group['std_scale']))
            else:
                plain.append(group)
        self._means_into(plain, with_grads=False)
        # the noise is drawn inside, in list order = param_group order
        _curv.sample_all(drawn)

    @staticmethod
    def _means_into(groups, with_grads):
        to, source = [], []
        for group in groups:
            for p, m in zip(group['params'], group['mean']):
                to.append(p.data)
                source.append(m.data)
                if with_grads and p.grad is not None and m.grad is not None:
                    to.append(p.grad)
                    source.append(m.grad)
        if to:
            torch._foreach_copy_(to, source)     # (one launch instead of one per tensor)

    def copy_mean_to_params(self):
        self._means_into(self.param_groups, with_grads=True)

    # ---- KL weighting --------------------------------------------------------------

    def adjust_kl_weighting(self):
        """Moves the l2 coefficient and the posterior scale of the groups that have
        them along the warm-up of the KL weight (reference: vi.py:150-172)."""
        warmup_steps = self.defaults['warmup_kl_weighting_steps']
        step = self.optim_state['step']
        if warmup_steps is None or step > warmup_steps:
            return
        rate = kl_rate(step, warmup_steps, self.defaults['warmup_kl_weighting_init'],
                       self.defaults['kl_weighting'])
        for group in self.param_groups:
            if group['l2_reg'] > 0:
                group['l2_reg'] = rate * self.defaults['l2_reg']
            if group['std_scale'] > 0:
                group['std_scale'] = math.sqrt(rate) * self.defaults['std_scale']

    # ---- step ----------------------------------------------------------------------

    def step(self, closure=None):
        """One VI step.  `closure` runs forward/backward and returns (loss, output).
        Returns (mean loss over the MC samples, accumulated probabilities)."""
        samples = self.defaults['num_mc_samples']
        micro = self.defaults['acc_steps']
        self.set_random_seed()

        loss_mean = prob_sum = None
        self._begin_accumulation(1 / samples / micro)
        try:
            for _ in range(samples):
                self.sample_params()
                loss, output = closure()
                loss_mean = _running_sum(loss_mean, loss.detach(), 1 / samples)
                # weight 1/acc_steps, not 1/samples: what the reference returns (vi.py:209)
                prob_sum = _running_sum(prob_sum, class_probabilities(output), 1 / micro)
                self._accumulate(1 / samples / micro)
        finally:
            # the hooks add to the accumulators during this loop only (the reference adds
            # curv.data inside its MC loop, vi.py:211-220): a forward pass that the caller
            # runs between two micro-steps, or after a closure that raised, must not
            self._end_accumulation()

        self.optim_state['acc_step'] += 1
        if self.optim_state['acc_step'] < micro:
            return loss_mean, prob_sum
        self.optim_state['acc_step'] = 0

        # the averages become the gradients of the means and the curvature data
        self.backward_postprocess(target='mean')
        self.optim_state['step'] += 1
        groups = self.local_param_groups
        self._update_groups(groups, target='mean', update_inv=True,
                            update_std=self._sampled(groups), precondition=True)
        self._means_into(groups, with_grads=True)
        self.adjust_kl_weighting()
        return loss_mean, prob_sum

    # ---- prediction ----------------------------------------------------------------

    def prediction(self, data, mc=None, keep_probs=False):
        """Predictive probabilities averaged over posterior samples (`mc` draws, default
        `val_num_mc_samples`; 0: the posterior mean alone); with `keep_probs` also the
        list of per-sample probabilities.  The parameters are the means again afterwards
        (reference: vi.py:260-299)."""
        self.set_random_seed(self.optim_state['step'])
        draws = self.defaults['val_num_mc_samples'] if mc is None else mc
        passes = max(draws, 1)
        average, kept = None, []
        for _ in range(passes):
            if draws == 0:
                self.copy_mean_to_params()
            else:
                self.sample_params()
            prob = class_probabilities(self.model(data))
            average = _running_sum(average, prob, 1 / passes)
            if keep_probs:
                kept.append(prob)
        self.copy_mean_to_params()
        return (average, kept) if keep_probs else average


class VOGN(VIOptimizer):
    """Variational online Gauss-Newton: VIOptimizer with diagonal curvature for
    every layer type (reference preset: optim/vi.py:302-319)."""

    PRESET = dict(lr=1e-3, curv_type='Cov',
                  curv_shapes={name: 'Diag' for name in
                               ('Linear', 'Conv2d', 'BatchNorm1d', 'BatchNorm2d')},
                  curv_kwargs={'ema_decay': 0.01, 'damping': 1e-7},
                  warmup_kl_weighting_init=0.01, warmup_kl_weighting_steps=1000,
                  grad_ema_decay=0.1, num_mc_samples=50, val_num_mc_samples=100)

    def __init__(self, *args, **kwargs):
        super(VOGN, self).__init__(*args, **dict(self.PRESET, **kwargs))
