"""The Phase-2 and Phase-1 elementwise kernels in the forms their dispatch
chooses (wide, strip and masked tiles, flat chunks; fp32 / bf16 / fp16; rows
that start at any element) against the CPU oracle from the same state."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import scao_amd
from oracle import scao_ref as R
from parity import kron_leaves

pytestmark = pytest.mark.gpu

# k, shapes: widths on both sides of the tiles of each kernel (16 x 256 wide;
# 64 x 128 and 128 x 64 strips; 64 x 64 masked), odd row strides, chunks of 4096
CASES = [(64, [(32, 512), (33, 257), (17, 300)]), (128, [(64, 256), (129, 385)]),
         (256, [(512, 512), (300, 515)]), (320, [(640, 700)]), (24, [(65, 1003), (4097,), (5,)]),
         (320, [(400, 515)])]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lars", [1e-3, 0.0])
@pytest.mark.parametrize("sparsity", [0.0, 0.7])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_phase2_step_forms(hip_device, dtype, lars, sparsity, case):
    """p and the moments after one step from the same random state.  fp32:
    the sums round differently, 1e-5 in the 2-norm; 16-bit types: the
    preconditioned gradient is rounded to the type twice, so an element next
    to a border may differ by 2^-8 (bf16) of itself -- in the 2-norm at most
    2^-8 if every element did."""
    k, shapes = CASES[case]
    g = torch.Generator().manual_seed(case)
    cfg = dict(lr=1e-3, lars_coeff=lars, k_min=k, k_max=k, warmup_steps=0, blend_steps=0,
               min_precond_updates=0, precond_freq=10 ** 9, max_precond_dim=1024,
               sparsity=sparsity, noise_std_init=0.0, lookahead_k=0, async_precond=False)
    init = [(0.02 * torch.randn(*s, generator=g)).to(dtype) for s in shapes]
    rp = [torch.nn.Parameter(x.clone()) for x in init]
    gp = [torch.nn.Parameter(x.clone().to(hip_device)) for x in init]
    ref, opt = R.RefSCAO(rp, **cfg), scao_amd.SCAO(gp, **cfg)
    for a, b in zip(rp, gp):
        ref._init_state(a, ref.param_groups[0])
        opt._init_state(b, opt.param_groups[0])
        sa, sb = ref.state[a], opt.state[b]
        for key, scale in (("exp_avg", 1e-5), ("exp_avg_diff", 1e-5), ("prev_grad", 1e-3)):
            sa[key].copy_(scale * torch.randn(a.shape, generator=g))
        sa["exp_avg_sq"].copy_(1e-9 * (0.1 + torch.rand(a.shape, generator=g)))
        for key in ("exp_avg", "exp_avg_sq", "exp_avg_diff", "prev_grad"):
            sb[key].copy_(sa[key])
        if a.ndim == 1:
            sa["preconditioner"].diag_ema.copy_(1e-6 * (0.1 + torch.rand(a.shape, generator=g)))
            sb["preconditioner"].diag_ema.copy_(sa["preconditioner"].diag_ema)
        for (x, _, _), (y, _, _) in zip(kron_leaves(sa["preconditioner"]),
                                        sb["preconditioner"].leaves()):
            kk = x.U_l.shape[1]
            x.U_l = torch.randn(x.m, kk, generator=g) / x.m ** 0.5
            x.U_r = torch.randn(x.n, kk, generator=g) / x.n ** 0.5
            x.S_l, x.S_r = (1e-3 * (0.1 + torch.rand(kk, generator=g)) for _ in range(2))
            for name in ("U_l", "U_r", "S_l", "S_r"):
                setattr(y, name, getattr(x, name).to(hip_device))
            y._touch()
        a.grad = (1e-3 * torch.randn(a.shape, generator=g)).to(dtype)
        b.grad = a.grad.to(hip_device)
    ref.step()
    opt.step()
    torch.cuda.synchronize()
    tol = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for a, b, x in zip(rp, gp, init):
        for key in ("exp_avg", "exp_avg_sq", "exp_avg_diff", "prev_grad"):
            want, got = ref.state[a][key].double(), opt.state[b][key].cpu().double()
            err = ((got - want).norm() / want.norm()).item()
            assert err < tol, (tuple(a.shape), key, err)
        du, dw = b.detach().cpu().double() - x.double(), a.detach().double() - x.double()
        # the update itself, up to one spacing of the stored parameter per
        # element: at most 2^-7 (bf16) of the larger of its old and new values
        # (an update may carry it into the next binade, where the grid doubles)
        eps = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
        size = torch.maximum(x.double().abs(), a.detach().double().abs()).clamp_min(2.0 ** -14)
        bound = eps * size * 1.01 + 2e-4 * dw.abs().max()
        bad = ((du - dw).abs() / bound).max().item()
        assert bad <= 1.0, (tuple(a.shape), bad)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("numel,off", [(4096, 0), (4095, 0), (4097, 1), (8192 + 5, 3), (3, 1)])
def test_phase1_chunks_at_any_element(hip_device, dtype, numel, off):
    """Warm-up steps of a parameter whose storage starts ``off`` elements into
    a buffer equal, bit for bit, those of an aligned copy."""
    g = torch.Generator().manual_seed(numel)
    base = (0.02 * torch.randn(numel + off, generator=g)).to(dtype).to(hip_device)
    pa = torch.nn.Parameter(base[off:])
    pb = torch.nn.Parameter(base[off:].clone())
    cfg = dict(warmup_steps=100, sparsity=0.0, noise_std_init=0.0, lookahead_k=0)
    oa, ob = scao_amd.SCAO([pa], **cfg), scao_amd.SCAO([pb], **cfg)
    for t in range(3):
        x = (1e-3 * torch.randn(numel + off, generator=g)).to(dtype).to(hip_device)
        pa.grad, pb.grad = x[off:], x[off:].clone()
        oa.step()
        ob.step()
    torch.cuda.synchronize()
    assert torch.equal(pa, pb)
    for key in ("exp_avg", "exp_avg_sq", "prev_grad"):
        assert torch.equal(oa.state[pa][key], ob.state[pb][key])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("phase2", [False, True])
def test_flat_tasks_do_not_read_b(hip_device, monkeypatch, dtype, phase2):
    """The Adam and LARS-write tasks are whole chunks whatever their second
    coordinate holds (a quarter's number is the diagonal kernels' alone): the
    step equals, bit for bit, the one with zeros there."""
    from scao_amd import engine as E
    g = torch.Generator().manual_seed(5)
    init = [(0.02 * torch.randn(*s, generator=g)).to(dtype).to(hip_device)
            for s in ((4096 * 3 + 5,), (100, 130))]
    grads = [(1e-3 * torch.randn(x.shape, generator=g)).to(dtype).to(hip_device) for x in init]
    cfg = dict(warmup_steps=0 if phase2 else 100, min_precond_updates=0, precond_freq=10 ** 9,
               sparsity=0.0, noise_std_init=0.0, lookahead_k=0, k_min=8, k_max=8)
    plain = E._param_tasks

    def marked(*args):
        arrays, *rest = plain(*args)
        arrays = {kind: arr.copy() for kind, arr in arrays.items()}
        for kind in ("adam", "lars"):
            if kind in arrays:
                arrays[kind][:, 2] = 1 + np.arange(len(arrays[kind])) % 7
        return (arrays, *rest)

    def run():
        ps = [torch.nn.Parameter(x.clone()) for x in init]
        opt = scao_amd.SCAO(ps, **cfg)
        for p, x in zip(ps, grads):
            p.grad = x
        opt.step()
        torch.cuda.synchronize()
        return [[p.detach()] + [opt.state[p][key] for key in
                                ("exp_avg", "exp_avg_sq", "exp_avg_diff", "prev_grad")] for p in ps]

    want = run()
    monkeypatch.setattr(E, "_param_tasks", marked)
    for a, b in zip(run(), want):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_norm_average_is_taken_once(hip_device):
    """scao_step_finalize's phase 1 takes the grad-norm average only when it is
    asked for with SCAO_NORM_EMA_PHASE1: a caller that passes its flag to both
    phases (and no runtime to the second) gets one update."""
    from scao_amd import _lib as L
    desc = np.zeros(1, dtype=L.PARAM_DESC)
    desc["pre_end"] = desc["post_end"] = 1
    desc["flags"] = L.PF_NORM
    params = L.upload(desc, hip_device)
    slots = torch.tensor([4.0, 1.0, 1.0], dtype=torch.float64, device=hip_device)   # ||g|| = 2
    stat = torch.zeros(L.PARAM_STAT.itemsize, dtype=torch.uint8, device=hip_device)
    runtime = torch.tensor([1.0, 0.0], dtype=torch.float64, device=hip_device)
    s = L.stream_ptr(hip_device)

    def finalize(rt, phase, flag):
        L.call("scao_step_finalize", params.data_ptr(), 1, slots.data_ptr(), stat.data_ptr(), rt,
               phase, flag, 1, s)
        return runtime.tolist()

    once = 0.95 * 1.0 + 0.05 * 2.0
    assert finalize(runtime.data_ptr(), 0, 1) == [once, 2.0]
    assert finalize(0, 1, 1) == [once, 2.0]
    assert finalize(runtime.data_ptr(), 1, 1) == [once, 2.0]
    assert finalize(runtime.data_ptr(), 1, L.NORM_EMA_PHASE1) == [0.95 * once + 0.05 * 2.0, 2.0]
    with pytest.raises(L.ScaoLibError):
        finalize(0, 1, L.NORM_EMA_PHASE1)
    with pytest.raises(L.ScaoLibError):
        finalize(0, 0, 1)
