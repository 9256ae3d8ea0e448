"""The step with gradient noise (the optimizer's default for its first
thousands of steps) through every apply kernel that forms it: wide, strip,
pipelined and masked tiles and flat chunks, fp32 / bf16 / fp16, with and
without the filter, rows that start at any element."""

from __future__ import annotations

import pytest
import torch

import scao_amd

pytestmark = pytest.mark.gpu

LR, WD, LARS = 1e-3, 0.01, 1e-3
# eps beside the gradients' size: the update stays a smooth function of them
BETA1, BETA2, BETA3, EPS = 0.9, 0.999, 0.99, 1e-4
SHAPES = [(512, 515), (256, 768), (100, 37), (4096 + 5,)]


def _make(dtype, k, sparsity, noise, phase2, dev):
    g = torch.Generator().manual_seed(k)
    params = [torch.nn.Parameter((0.02 * torch.randn(s, generator=g)).to(dtype).to(dev))
              for s in SHAPES]
    grads = [(1e-3 * torch.randn(s, generator=g)).to(dtype).to(dev) for s in SHAPES]
    sched = (dict(warmup_steps=0, min_precond_updates=0, blend_steps=0) if phase2
             else dict(warmup_steps=10))
    opt = scao_amd.SCAO(params, lr=LR, weight_decay=WD, lars_coeff=LARS, betas=(BETA1, BETA2),
                        beta3=BETA3, eps=EPS, sparsity=sparsity, noise_std_init=noise,
                        lookahead_k=0, precond_freq=10 ** 9, k_min=k, k_max=k,
                        max_precond_dim=1024, **sched)
    for p, x in zip(params, grads):
        opt._init_state(p, opt.param_groups[0])
        pre = opt.state[p]["preconditioner"]
        if p.ndim == 1:
            pre.diag_ema.copy_(1e-6 * (0.1 + torch.rand(p.shape, generator=g)))
        for leaf, _, _ in pre.leaves():
            kk = leaf.U_l.shape[1]
            leaf.U_l = (torch.randn(leaf.m, kk, generator=g) / leaf.m ** 0.5).to(dev)
            leaf.U_r = (torch.randn(leaf.n, kk, generator=g) / leaf.n ** 0.5).to(dev)
            leaf.S_l, leaf.S_r = ((1e-3 * (0.1 + torch.rand(kk, generator=g))).to(dev)
                                  for _ in range(2))
            leaf._touch()
        p.grad = x
    return params, grads, opt


# apply variants that a step of this rank takes with moments of their own (bit
# 1) and LARS (bit 2): wide (4), pipelined (8; fp32 only), strip (16; 32: k =
# 128), and their 16-bit forms (64); at 320 the 256-row parameter keeps rank 256
VARIANTS = {64: {7, 3}, 128: {55, 3}, 256: {23, 3}, 320: {15, 23, 3}}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [64, 128, 256, 320])
@pytest.mark.parametrize("sparsity", [0.0, 0.7])
def test_noisy_phase2_step(hip_device, dtype, k, sparsity):
    """The moment gradient (stored as prev_grad) equals, bit for bit, what the
    filter's output pass writes for the same state and noise key.  The
    preconditioned gradient does not see noise or filter, so exp_avg is that of
    a step without them, and the other moments and the update follow from the
    two in float64: 1e-5 in the 2-norm (fp32 sums), or 2^-8 / 2^-11 where the
    preconditioned gradient is rounded to a 16-bit type."""
    from scao_amd import engine
    from scao_amd.optimizer import _SparseGradFilter
    noise = 0.01
    params, grads, opt = _make(dtype, k, sparsity, noise, True, hip_device)
    plain, _, ref = _make(dtype, k, 0.0, 0.0, True, hip_device)
    before = [p.detach().double() for p in params]
    torch.manual_seed(11)
    opt.step()
    ref.step()
    want = VARIANTS[k]
    if dtype != torch.float32:
        want = {v + 64 if v & 4 else v for v in want if not v & 8}
    assert want == {int(v[5:]) for v, n in opt._ws.ntasks.items() if v.startswith("apply") and n}
    filters = [_SparseGradFilter(sparsity) if sparsity else None for _ in SHAPES]
    torch.manual_seed(11)
    formed = engine.moment_grads(list(zip(filters, grads)), noise)
    torch.cuda.synchronize()
    tol = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]

    def close(got, exp, what):
        err = ((got.double() - exp).norm() / exp.norm()).item()
        assert err < tol, (what, err)

    for p, q, gm, p0 in zip(params, plain, formed, before):
        st = opt.state[p]
        assert torch.equal(st["prev_grad"], gm), tuple(p.shape)
        m = ref.state[q]["exp_avg"].double()
        close(st["exp_avg"], m, "exp_avg")
        gp, d = m / (1 - BETA1), gm.double()
        close(st["exp_avg_diff"], (1 - BETA3) * d, "exp_avg_diff")
        v = (1 - BETA2) * (gp + (1 - BETA3) * d).square()
        close(st["exp_avg_sq"], v, "exp_avg_sq")
        # first step: the bias corrections are 1 - beta
        u = (gp + (1 - BETA3) * d) / ((v / (1 - BETA2)).sqrt() + EPS)
        pd = p0 * (1 - LR * WD)
        trust = LARS * pd.norm() / (u.norm() + WD * pd.norm() + 1e-8)
        exp = pd - LR * trust * u
        # the update itself, up to a spacing of the stored parameter (fp32: the
        # decay factor, its product and the sum each round by half of one) and
        # the tolerance of u's denominator
        eps = {torch.float32: 1.5 * 2.0 ** -23, torch.bfloat16: 2.0 ** -7,
               torch.float16: 2.0 ** -10}[dtype]
        bound = 1.01 * eps * exp.abs().clamp_min(2.0 ** -14) + 4 * tol * LR * trust * u.abs().max()
        bad = ((p.detach().double() - exp).abs() / bound).max().item()
        assert bad <= 1.0, (tuple(p.shape), bad)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sparsity", [0.0, 0.7])
def test_noisy_warm_up_step(hip_device, dtype, sparsity):
    """Phase 1: the moment gradient bit for bit, and exp_avg its (1 - beta1)
    multiple."""
    from scao_amd import engine
    from scao_amd.optimizer import _SparseGradFilter
    params, grads, opt = _make(dtype, 64, sparsity, 0.01, False, hip_device)
    torch.manual_seed(5)
    opt.step()
    filters = [_SparseGradFilter(sparsity) if sparsity else None for _ in SHAPES]
    torch.manual_seed(5)
    formed = engine.moment_grads(list(zip(filters, grads)), 0.01)
    torch.cuda.synchronize()
    for p, gm in zip(params, formed):
        st = opt.state[p]
        assert torch.equal(st["prev_grad"], gm), tuple(p.shape)
        assert torch.allclose(st["exp_avg"], (1 - BETA1) * gm, rtol=1e-6, atol=0.0)
        assert torch.allclose(st["exp_avg_sq"], (1 - BETA2) * gm * gm, rtol=1e-5, atol=1e-30)
