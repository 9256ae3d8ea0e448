"""Two large dense factors of one dimension: the batched solver in place of
the library (engine.batch_route), through the refresh."""

import pytest
import torch

from scao_amd import SparsePreconditioner, engine

K = 64


def _planted(n, gen):
    """(Q, X): X symmetric with eigenvalues 1 .. 0.5 on Q's columns and at most
    0.05 on the rest of the space."""
    Q, _ = torch.linalg.qr(torch.randn(n, K, generator=gen, dtype=torch.float64))
    lam = 1.0 - torch.arange(K, dtype=torch.float64) / (2 * K)
    B = torch.randn(n, 2 * K, generator=gen, dtype=torch.float64)
    B -= Q @ (Q.T @ B)
    B *= (0.05 ** 0.5) / torch.linalg.matrix_norm(B, 2)
    X = ((Q * lam) @ Q.T + B @ B.T).float()
    return Q, 0.5 * (X + X.T)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2048, 2064, 3072])
def test_pair_takes_the_solver(n, monkeypatch):
    dev = torch.device("cuda:0")
    gen = torch.Generator().manual_seed(n)
    (Ql, Xl), (Qr, Xr) = _planted(n, gen), _planted(n, gen)
    kw = dict(k_min=K, k_max=K, max_precond_dim=4096, use_int8_ema=False)
    got = {}
    for route in ("hip", "library"):
        if route == "library":
            monkeypatch.setattr(engine, "batch_route", lambda r, dim, count: "library")
        pre = SparsePreconditioner(torch.zeros(n, n, device=dev), **kw)
        pre.precond_step = 4
        pre.L_ema, pre.R_ema = Xl.to(dev), Xr.to(dev)
        print(f"n={n} {route}", flush=True)
        engine.refresh([(pre, torch.zeros(n, n, device=dev))], eigen_only=True)
        torch.cuda.synchronize()
        assert engine.LAST_REFRESH_ROUTES == {route: 2}
        got[route] = pre
    # a float32 solver's backward error is at most n eps |X| (|X| = 1, the
    # debiasing scales both sides alike); it turns the wanted space by that over
    # its gap of 0.45 to the rest and moves a value of at least 0.5 by that
    bound = n * 2.0 ** -24
    a, b = got["hip"], got["library"]
    assert a.k == b.k == K
    for Q, U, S, Sb in ((Ql, a.U_l, a.S_l, b.S_l), (Qr, a.U_r, a.S_r, b.S_r)):
        U, S, Sb = U.double().cpu(), S.double().cpu(), Sb.double().cpu()
        assert torch.linalg.matrix_norm(U - Q @ (Q.T @ U), 2) <= bound / 0.45
        assert ((S - Sb).abs() / Sb).max() <= 2 * bound / 0.5   # one error a side
        assert (U.T @ U - torch.eye(K, dtype=torch.float64)).abs().max() <= bound


def test_pair_route():
    for n in (2048, 2064, 3072, 4080):
        assert engine.batch_route("hip", n, 1) == "library"
        assert engine.batch_route("hip", n, 2) == "hip"
    for n in (16, 2032):
        assert engine.batch_route("hip", n, 1) == "hip"
    assert engine.batch_route("library", 2048, 2) == "library"
