"""The projection and delta stages in the forms their dispatch chooses: whole
and masked tiles, fp32 / bf16 / fp16 data, rows that start at any element,
row parts and column chunks, against float64."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import scao_amd

pytestmark = pytest.mark.gpu


def _rand(gen, *s):
    return torch.randn(*s, generator=gen)


# (m, n, k, row stride): tile edges on both sides of 32 rows, 256 columns and
# ranks 64 / 128 / 256; one to 16 row parts; a tiny block with no room for planes
OP_SHAPES = [(32, 256, 64, 256), (33, 257, 64, 257), (31, 255, 63, 300), (127, 300, 33, 301),
             (256, 256, 65, 259), (1000, 513, 100, 513), (640, 1024, 128, 1025),
             (513, 700, 129, 700), (512, 512, 256, 512), (300, 1000, 257, 1003),
             (2048, 2048, 64, 2048), (4096, 96, 64, 96), (7, 5, 3, 5), (2, 300, 2, 301)]


@pytest.mark.parametrize("m,n,k,ld", OP_SHAPES)
@pytest.mark.parametrize("inplace", [False, True])
def test_fused_operator_forms(hip_device, m, n, k, ld, inplace):
    """out against float64, elementwise relative to the absolute sums it is
    made of (each product within 2^-23, sums of at most 4096 + 256 + 256 fp32
    terms in partial sums of a few hundred: 2e-5 covers them); in place (out
    is G) no planes fit, the same tolerance."""
    from scao_amd import _lib as L
    g = torch.Generator().manual_seed(m + 3 * n + 7 * k)
    U_l, U_r = _rand(g, m, k) / m ** 0.5, _rand(g, n, k) / n ** 0.5
    s_l, s_r = torch.rand(k, generator=g) * 3 + 0.1, torch.rand(k, generator=g) * 3 + 0.1
    G = _rand(g, m, ld)
    dev = [t.to(hip_device) for t in (U_l, s_l, U_r, s_r, G)]
    if inplace and ld != n:
        pytest.skip("out is m x n without a row stride")
    ws = torch.empty(L.lib().scao_fused_kronecker_workspace(m, n, k) // 4, device=hip_device)
    out = dev[4] if inplace else torch.full((m, n), float("nan"), device=hip_device)
    L.call("scao_fused_kronecker_precond", *[t.data_ptr() for t in dev], ld, out.data_ptr(), m, n,
           k, ws.data_ptr(), L.stream_ptr(hip_device))
    a, b, x = U_l.double(), U_r.double(), G[:, :n].double()
    f = s_l.double()[:, None] * s_r.double() - 1.0
    want = x + a @ (f * (a.T @ x @ b)) @ b.T
    scale = x.abs() + a.abs() @ (f.abs() * (a.abs().T @ x.abs() @ b.abs())) @ b.abs().T
    err = ((out.cpu().double() - want).abs() / scale).max().item()
    assert err < 2e-5, err


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("shared", ["U_l", "s_l", "s_r"])
@pytest.mark.parametrize("m,n,k", [(512, 512, 64), (1000, 513, 100)])
def test_fused_operator_out_shares_an_operand(hip_device, m, n, k, shared, noalloc):
    """An out that takes the storage of an operand that only the first stages
    read, at its first and at its last floats: no partial sums go there while
    the operand is still read.  Tolerance as above."""
    from scao_amd import _lib as L
    g = torch.Generator().manual_seed(m + k)
    ops = dict(U_l=_rand(g, m, k) / m ** 0.5, s_l=torch.rand(k, generator=g) * 3 + 0.1,
               U_r=_rand(g, n, k) / n ** 0.5, s_r=torch.rand(k, generator=g) * 3 + 0.1,
               G=_rand(g, m, n))
    a, b, x = ops["U_l"].double(), ops["U_r"].double(), ops["G"].double()
    f = ops["s_l"].double()[:, None] * ops["s_r"].double() - 1.0
    want = x + a @ (f * (a.T @ x @ b)) @ b.T
    scale = x.abs() + a.abs() @ (f.abs() * (a.abs().T @ x.abs() @ b.abs())) @ b.abs().T
    for at_end in (False, True):
        dev = {name: t.to(hip_device) for name, t in ops.items()}
        out = torch.empty(m, n, device=hip_device)
        t = dev[shared]
        part = out.view(-1)[-t.numel():] if at_end else out.view(-1)[:t.numel()]
        dev[shared] = part.view(t.shape).copy_(t)
        ptrs = [dev[name].data_ptr() for name in ("U_l", "s_l", "U_r", "s_r", "G")]
        ws = torch.empty(L.lib().scao_fused_kronecker_workspace(m, n, k) // 4, device=hip_device)
        name = "scao_fused_kronecker_precond" + ("_noalloc" if noalloc else "")
        L.call(name, *ptrs, n, out.data_ptr(), m, n, k, *([] if noalloc else [ws.data_ptr()]),
               L.stream_ptr(hip_device))
        err = ((out.cpu().double() - want).abs() / scale).max().item()
        assert err < 2e-5, (shared, at_end, err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shapes,k", [([(96, 300), (257, 511)], 64), ([(1000, 1537)], 40),
                                      ([(640, 768), (129, 257)], 128), ([(512, 520)], 256),
                                      ([(2048, 2048)], 64), ([(64, 1024)] * 3, 24)])
def test_step_projection_and_delta(hip_device, dtype, shapes, k):
    """T = U_l^T G, Delta and the gradient norm of one Phase-2 step, read from
    the step's workspace, against float64 from the same factors."""
    from scao_amd import _lib as L
    g = torch.Generator().manual_seed(k)
    params = [torch.nn.Parameter((0.02 * _rand(g, *s)).to(dtype).to(hip_device)) for s in shapes]
    opt = scao_amd.SCAO(params, k_min=k, k_max=k, warmup_steps=0, min_precond_updates=0,
                        precond_freq=10 ** 9, max_precond_dim=1024, sparsity=0.0,
                        noise_std_init=0.0, lookahead_k=0, use_int8_ema=True)
    grads = [(1e-3 * _rand(g, *s)).to(dtype) for s in shapes]
    for p, x in zip(params, grads):
        p.grad = x.to(hip_device)
        opt._init_state(p, opt.param_groups[0])
        for leaf, _, _ in opt.state[p]["preconditioner"].leaves():
            kk = leaf.U_l.shape[1]
            leaf.U_l = (_rand(g, leaf.m, kk) / leaf.m ** 0.5).to(hip_device)
            leaf.U_r = (_rand(g, leaf.n, kk) / leaf.n ** 0.5).to(hip_device)
            leaf.S_l = torch.rand(kk, generator=g).add(0.1).to(hip_device)
            leaf.S_r = torch.rand(kk, generator=g).add(0.1).to(hip_device)
            leaf._touch()
    opt.step()
    torch.cuda.synchronize()
    ws = opt._ws
    scratch = ws._bufs["leaf_scratch"]
    flat = scratch.view(torch.float32)
    tab = np.frombuffer(ws.leaf_dev.cpu().numpy().tobytes(), dtype=L.LEAF_DESC)

    def read(ptr, *s):
        o = (int(ptr) - scratch.data_ptr()) // 4
        return flat[o:o + s[0] * s[1]].view(*s).double().cpu()

    nblk = 0
    for (leaf, r0, c0, pi), e in zip(ws.leaves, tab):
        if not leaf.use_kronecker:
            continue
        m, n, kp, kk = int(e["m"]), int(e["n"]), int(e["k"]), leaf.U_l.shape[1]
        G = grads[pi][r0:r0 + m, c0:c0 + n].double()
        U, V = leaf.U_l.double().cpu(), leaf.U_r.double().cpu()
        T, D = read(e["T"], kp, n), read(e["Delta"], kp, kp)
        err = ((T[:kk] - U.T @ G).abs() / (U.abs().T @ G.abs())).max().item()
        assert err < 1e-5, (m, n, err)
        f = (leaf.S_l.double().cpu()[:, None] * leaf.S_r.double().cpu()).pow(-0.25) - 1.0
        big = (f.abs() + 1.0) * (U.abs().T @ G.abs() @ V.abs())   # s_l s_r - 1 cancels near 1
        err = ((D[:kk, :kk] - f * (U.T @ G @ V)).abs() / big).max().item()
        assert err < 1e-5, (m, n, err)
        assert not T[kk:].any() and not D[kk:].any() and not D[:, kk:].any()
        nblk += 1
    assert nblk
    stat = ws._bufs["stat"].cpu().numpy().tobytes()[:len(params) * L.PARAM_STAT.itemsize]
    for x, st in zip(grads, np.frombuffer(stat, dtype=L.PARAM_STAT)):
        want = x.double().square().sum().item()
        assert abs(float(st["g2"]) - want) <= 1e-6 * want


def test_cut_of_the_sums_changes_rounding_only(hip_device):
    """A step cuts the sums of its projection and delta stages by how many
    blocks it has, so a parameter steps with other roundings alone than beside
    308 blocks more: 1e-6 in the 2-norm of its moments (an fp32 sum of 512
    terms, in one chain or in parts, is within 2^-24 times a few of 512^0.5 of
    it), and the same bits each time in the same company."""
    from scao_amd import engine as E
    g = torch.Generator().manual_seed(2)
    init = [0.02 * _rand(g, 512, 512), 0.02 * _rand(g, 308 * 256, 256)]
    grads = [1e-3 * _rand(g, *x.shape) for x in init]
    factors = [_rand(g, 256, 64) / 16.0 for _ in range(8)]
    spectra = [1e-3 * (0.1 + torch.rand(64, generator=g)) for _ in range(8)]

    def run(n):
        params = [torch.nn.Parameter(x.to(hip_device)) for x in init[:n]]
        opt = scao_amd.SCAO(params, k_min=64, k_max=64, warmup_steps=0, min_precond_updates=0,
                            precond_freq=10 ** 9, max_precond_dim=256, sparsity=0.0,
                            noise_std_init=0.0, lookahead_k=0, blend_steps=0)
        for p, x in zip(params, grads):
            p.grad = x.to(hip_device)
            opt._init_state(p, opt.param_groups[0])
        for i, (leaf, _, _) in enumerate(opt.state[params[0]]["preconditioner"].leaves()):
            leaf.U_l, leaf.U_r = (factors[2 * i + j].to(hip_device) for j in range(2))
            leaf.S_l, leaf.S_r = (spectra[2 * i + j].to(hip_device) for j in range(2))
            leaf._touch()
        opt.step()
        torch.cuda.synchronize()
        st = opt.state[params[0]]
        plan = E._split_plan([lf for lf, *_ in opt._ws.leaves])
        return plan, [params[0].detach()] + [st[key] for key in
                                             ("exp_avg", "exp_avg_sq", "exp_avg_diff")]

    alone, few = run(1)
    beside, many = run(2)
    assert alone.rows and alone.chunks and not beside.rows and not beside.chunks
    for a, b in zip(few, many):
        assert ((a - b).double().norm() / a.double().norm()).item() < 1e-6
    for n, first in ((1, few), (2, many)):
        assert all(torch.equal(a, b) for a, b in zip(first, run(n)[1]))
