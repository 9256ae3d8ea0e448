"""The work that a user of scao_amd has it do, as cases that can be timed.

Four kinds of case, each through an entry point that a program calls:

  step     one ``scao_amd.SCAO.step()`` without a curvature refresh: Phase 2
           (preconditioned Adan, what almost every step of a run is) or Phase 1
           (Adam, the warm-up), from a training run's state;
  refresh  one ``SCAO.step()`` that also refreshes the curvature: Gram product,
           EMA, requantisation, eigenfactors, then the step with them;
  fused    ``scao_amd.hip.fused_kronecker_precond`` on one block;
  ema      ``scao_amd.hip.int8_ema_update`` on one factor.

``shapes`` lists parameters as "2048x8192*2,2048": sizes joined by x, * for
several of one shape.  Everything is made on the GPU from the seed.
"""

import math

import torch

import scao_amd
from scao_amd import hip

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
LR, WD, EPS, TAU, LARS, RHO = 1e-3, 0.01, 1e-8, 1.0, 1e-3, 0.999
BETA1, BETA2, BETA3 = 0.9, 0.999, 0.99
FILTER_EMA = 0.99
# where in a run the state stands: parameter steps, Phase-2 steps, refreshes so far
STEP, SCAO_STEP, REFRESHES = 200, 60, 20

_LLAMA1B = "2048x2048*2,512x2048*2,8192x2048*2,2048x8192"
_GPT2S = "768x2304,768x768,768x3072,3072x768"


def listed():
    return [
        # the smallest model a user trains: one GPT-2-small layer with its
        # vectors, every parameter in one group.  Launches and latency.
        dict(name="step gpt2 layer", kind="step", phase=2, shapes=_GPT2S + ",768*4", dtype="fp32",
             k=64, dim=1024, sparsity=0.0),
        # the repository's headline model's embedding (63 blocks) and one
        # layer, all of it preconditioned, fp32 master weights
        dict(name="step llama1b embed+layer", kind="step", phase=2,
             shapes="128256x2048," + _LLAMA1B + ",2048*3", dtype="fp32", k=64, dim=2048,
             sparsity=0.0),
        # the same layer held in bf16, as a model loaded in its checkpoint's
        # type is trained
        dict(name="step llama1b layer bf16", kind="step", phase=2, shapes=_LLAMA1B + ",2048*2",
             dtype="bf16", k=64, dim=2048, sparsity=0.0),
        # one Qwen-3B layer with the optimizer's default gradient filter and
        # rank: the moments see another gradient than the preconditioner
        dict(name="step qwen3b layer filter", kind="step", phase=2,
             shapes="2048x2048*2,256x2048*2,11008x2048*2,2048x11008,2048*2", dtype="fp32", k=128,
             dim=2048, sparsity=0.7),
        # one Llama-8B layer: the largest blocks and the largest rank
        dict(name="step llama8b layer", kind="step", phase=2,
             shapes="4096x4096*2,1024x4096*2,14336x4096*2,4096x14336,4096*2", dtype="fp32", k=256,
             dim=4096, sparsity=0.0),
        # sizes that no tile divides: odd rows and columns, a convolution, a
        # remainder block one column wide, a rank between the kernels' widths
        dict(name="step odd sizes", kind="step", phase=2,
             shapes="1000x1537,513x2049,2049x1003,256x128x3x3,50x333,1001", dtype="fp32", k=40,
             dim=1024, sparsity=0.0),
        # warm-up: the Adam steps that every run begins with, bf16 weights
        dict(name="warm-up llama1b bf16", kind="step", phase=1,
             shapes="128256x2048," + _LLAMA1B + ",2048*3", dtype="bf16", k=64, dim=2048,
             sparsity=0.0),
        # refresh whose int8 EMAs stay exactly diagonal: small gradients
        # (N(0, 1e-3^2)), the attention and down projections of Llama-1B
        dict(name="refresh llama1b diagonal", kind="refresh", shapes="2048x2048*2,512x2048,2048x8192",
             dtype="fp32", k=64, dim=2048, ema="int8", spectrum="diagonal"),
        # refresh whose EMAs are dense (gradients of low rank plus noise): the
        # same projections through the eigensolver
        dict(name="refresh llama1b dense", kind="refresh", shapes="2048x2048*2,512x2048,2048x8192",
             dtype="fp32", k=64, dim=2048, ema="int8", spectrum="dense"),
        # refresh of a small model with fp32 EMAs (the sub-1B preset), with
        # remainder blocks and a vector
        dict(name="refresh gpt2 layer fp32", kind="refresh", shapes="768x2304,768x768,768x3072,768",
             dtype="fp32", k=64, dim=1024, ema="fp32", spectrum="dense"),
        # the operator on one block, as the reference's maintainers bind it
        dict(name="fused 2048x2048", kind="fused", m=2048, n=2048, k=64, ld=2048),
        # the EMA operator on one factor
        dict(name="ema 4096x4096", kind="ema", rows=4096, cols=4096),
    ]


# ------------------------------------------------------------------ draw ---

def _size(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm; half of them whole
    multiples of 64, the others whatever comes, odd ones among them."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and v >= 64:
        v = v // 64 * 64
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "refresh", "fused", "ema"])
    if kind == "fused":
        m, n = _size(rng, 32, 4096), _size(rng, 32, 4096)
        k = rng.choice([8, 16, 33, 48, 64, 100, 128, 192, 256])
        pad = rng.choice([0, 0, 4, 512, 1001])
        return dict(kind="fused", m=m, n=n, k=min(k, m, n), ld=n + pad)
    if kind == "ema":
        return dict(kind="ema", rows=_size(rng, 32, 8192), cols=_size(rng, 32, 8192))
    if kind == "refresh":
        spectrum = rng.choice(["diagonal", "dense"])
        shapes, left = [], 12_000_000
        for _ in range(rng.randint(1, 3)):
            m, n = _size(rng, 64, 2048), _size(rng, 64, 4096)
            if m * n <= left:
                shapes.append("%dx%d" % (m, n))
                left -= m * n
        return dict(kind="refresh", shapes=",".join(shapes), dtype=rng.choice(["fp32", "bf16"]),
                    k=rng.choice([16, 32, 48, 64]), dim=rng.choice([1024, 2048]),
                    ema="int8" if spectrum == "diagonal" else rng.choice(["int8", "fp32"]),
                    spectrum=spectrum)
    shapes, left = [], 200_000_000
    for _ in range(rng.randint(1, 6)):
        m, n = _size(rng, 16, 16384), _size(rng, 16, 16384)
        if m * n <= left:
            shapes.append("%dx%d" % (m, n))
            left -= m * n
    shapes.append("%d" % _size(rng, 16, 16384))
    return dict(kind="step", phase=rng.choice([1, 2, 2, 2]), shapes=",".join(shapes),
                dtype=rng.choice(["fp32", "fp32", "bf16", "bf16", "fp16"]),
                k=rng.choice([8, 24, 48, 64, 100, 128, 256]), dim=rng.choice([1024, 2048, 4096]),
                sparsity=rng.choice([0.0, 0.0, 0.7]))


# ---------------------------------------------------------------- inputs ---

def _shapes(case):
    out = []
    for part in case["shapes"].split(","):
        one, _, many = part.partition("*")
        out += [tuple(int(x) for x in one.split("x"))] * int(many or 1)
    return out


def _blocks(shape, dim, r0=0, c0=0):
    """(m, n, row, column) of each block of a parameter's 2-D view."""
    m, n = shape
    if max(m, n) <= dim or min(m, n) <= 1:
        return [(m, n, r0, c0)]
    big, small = (m, n) if m >= n else (n, m)
    out = []
    for o in range(0, big, dim):
        b = min(dim, big - o)
        out += (_blocks((b, small), dim, r0 + o, c0) if m >= n
                else _blocks((small, b), dim, r0, c0 + o))
    return out


def _rank(m, n, k):
    """The rank a block of this size keeps with k_min = k_max = k."""
    d = min(m, n)
    return min(k, d // 2) if d > 2 * min(k, d) else min(k, d)


def _flat(shape):
    return (1, shape[0]) if len(shape) == 1 else (shape[0], math.prod(shape[1:]))


def _kron(m, n):
    return m > 1 and n > 1


def _orthonormal(gen, m, k):
    a = torch.randn(m, k, generator=gen, device=DEV, dtype=torch.float64)
    ch = torch.linalg.cholesky(a.T @ a)
    return torch.linalg.solve_triangular(ch, a.T, upper=False).T.float().contiguous()


def _codes(x):
    scale = float(x.abs().max()) / 127.0
    return (x / scale).round().clamp(-127, 127).to(torch.int8), scale


def _step_inputs(case, seed):
    """A training run's state at STEP, parameter by parameter, and two
    gradient sets, from the seed alone."""
    gen = torch.Generator(device=DEV).manual_seed(seed)

    def rnd(*s):
        return torch.randn(*s, generator=gen, device=DEV)

    dt, k, refresh = DTYPES[case["dtype"]], case["k"], case["kind"] == "refresh"
    dense = refresh and case["spectrum"] == "dense"
    sigma = 0.02 if dense else 1e-3
    out = []
    for shape in _shapes(case):
        m, n = _flat(shape)
        if dense and _kron(m, n):
            # a signal of rank k in fixed subspaces plus noise a tenth its size
            a, b = rnd(m, k) / math.sqrt(k), rnd(k, n)
            grads = []
            for _ in range(3):
                s = torch.linspace(1.0, 0.5, k, device=DEV) * torch.sign(rnd(k))
                grads.append(sigma * ((a * s) @ b + 0.1 * rnd(m, n)))
        else:
            grads = [sigma * rnd(m, n) for _ in range(3)]
        hist = grads[2]
        one = dict(shape=shape, p=(0.02 * rnd(m, n)).to(dt).reshape(shape),
                   grads=[g.to(dt).reshape(shape) for g in grads[:2]],
                   prev=hist.reshape(shape).clone(), hist=hist.to(dt).reshape(shape))
        mom = sigma if case.get("phase") == 1 else 0.01 * sigma
        one["exp_avg"] = (mom * rnd(m, n)).reshape(shape)
        one["exp_avg_sq"] = (mom * mom * (0.1 + torch.rand(m, n, generator=gen, device=DEV))
                             ).reshape(shape)
        one["exp_avg_diff"] = (mom * rnd(m, n)).reshape(shape)
        one["blocks"] = []
        for bm, bn, r, c in _blocks((m, n), case["dim"]):
            blk = dict(m=bm, n=bn, r=r, c=c)
            if _kron(bm, bn):
                kb = _rank(bm, bn, k)
                if refresh:
                    # the factors a refresh replaces
                    blk["U"] = [torch.eye(d, kb, device=DEV) for d in (bm, bn)]
                    blk["S"] = [torch.ones(kb, device=DEV) for _ in range(2)]
                    h = hist[r:r + bm, c:c + bn]
                    old = RHO ** REFRESHES
                    ema = []
                    for x in (h, h.T):
                        g = x @ x.T
                        g = g if dense else torch.diag(g.diagonal())
                        ema.append(g.mul_(1.0 - old).add_(
                            torch.eye(len(x), device=DEV), alpha=1e-4 * old))
                    blk["ema"] = [_codes(e) if case["ema"] == "int8" else e for e in ema]
                else:
                    blk["U"] = [_orthonormal(gen, d, kb) for d in (bm, bn)]
                    blk["S"] = [max(bm, bn) * sigma ** 2 * torch.logspace(0, -2, kb, device=DEV)
                                * (1 + 0.1 * torch.rand(kb, generator=gen, device=DEV))
                                for _ in range(2)]
            one["blocks"].append(blk)
        out.append(one)
    return out


def _optimizer(case, params):
    return scao_amd.SCAO(
        params, lr=LR, betas=(BETA1, BETA2), eps=EPS, weight_decay=WD, precond_freq=10 ** 9,
        k_min=case["k"], k_max=case["k"], rho=RHO, tau=TAU,
        warmup_steps=10 ** 9 if case.get("phase") == 1 else 0, blend_steps=50,
        min_precond_updates=0, max_precond_dim=case["dim"],
        use_int8_ema=case.get("ema", "int8") == "int8", async_precond=False, beta3=BETA3,
        sparsity=case.get("sparsity", 0.0), noise_std_init=0.0, lars_coeff=LARS, lookahead_k=0)


def _prepare_step(case, seed):
    inputs = _step_inputs(case, seed)
    params = [torch.nn.Parameter(one["p"].clone()) for one in inputs]
    opt = _optimizer(case, params)
    for p, one in zip(params, inputs):
        p.grad = one["hist"]
    opt.step()     # makes the state (and a filter's first average), replaced below
    for p, one in zip(params, inputs):
        p.data.copy_(one["p"])
        st = opt.state[p]
        for key, name in (("exp_avg", "exp_avg"), ("exp_avg_sq", "exp_avg_sq"),
                          ("exp_avg_diff", "exp_avg_diff"), ("prev_grad", "prev")):
            st[key].copy_(one[name])
        st["step"], st["scao_step"] = STEP, SCAO_STEP
        pre = st["preconditioner"]
        if case.get("phase") == 1:
            continue
        leaves = [leaf for leaf, _, _ in pre.leaves(diag=True)] or [pre]
        hist = one["hist"].reshape(_flat(one["shape"]))
        for leaf, blk in zip(leaves, one["blocks"]):
            if not _kron(blk["m"], blk["n"]):
                h = hist[blk["r"]:blk["r"] + blk["m"], blk["c"]:blk["c"] + blk["n"]]
                leaf.update_curvature(h.reshape(leaf.diag_ema.shape))
                leaf.precond_step = REFRESHES
                continue
            d = dict(precond_step=REFRESHES, k=blk["U"][0].shape[1], U_l=blk["U"][0],
                     U_r=blk["U"][1], S_l=blk["S"][0], S_r=blk["S"][1])
            if "ema" in blk:
                if case["ema"] == "int8":
                    (d["L_ema_q"], d["L_ema_scale"]), (d["R_ema_q"], d["R_ema_scale"]) = blk["ema"]
                else:
                    d["L_ema"], d["R_ema"] = blk["ema"]
            else:
                own = leaf.state_dict()
                d.update({n: own[n] for n in own if "ema" in n})
            leaf.load_state_dict(d)
        pre.precond_step = REFRESHES
    if case["kind"] == "refresh":
        for g in opt.param_groups:
            g["precond_freq"] = 1
    return dict(kind=case["kind"], opt=opt, params=params,
                grads=[[one["grads"][j] for one in inputs] for j in range(2)], at=0,
                int8=case.get("ema") == "int8")


def _matrix_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if case["kind"] == "fused":
        m, n, k = case["m"], case["n"], case["k"]
        wide = 1e-3 * torch.randn(m, case["ld"], generator=gen, device=DEV)
        s = [(max(m, n) * 1e-6 * torch.logspace(0, -2, k, device=DEV)
              * (1 + 0.1 * torch.rand(k, generator=gen, device=DEV))).pow(-0.25) for _ in range(2)]
        return dict(U_l=_orthonormal(gen, m, k), U_r=_orthonormal(gen, n, k), s_l=s[0], s_r=s[1],
                    G=wide[:, :n])
    r, c = case["rows"], case["cols"]
    x = torch.randn(r, c, generator=gen, device=DEV)
    q, scale = _codes(1e-4 * x)
    return dict(q=q, scale=scale, v=1e-7 * torch.randn(r, c, generator=gen, device=DEV))


def prepare(case, seed):
    if case["kind"] in ("step", "refresh"):
        return _prepare_step(case, seed)
    return dict(kind=case["kind"], **_matrix_inputs(case, seed))


# ------------------------------------------------------------------- run ---

def run(state):
    if state["kind"] == "fused":
        return hip.fused_kronecker_precond(state["U_l"], state["s_l"], state["U_r"], state["s_r"],
                                           state["G"])
    if state["kind"] == "ema":
        return hip.int8_ema_update(state["q"], state["scale"], state["v"], RHO)
    opt, params = state["opt"], state["params"]
    for p, g in zip(params, state["grads"][state["at"]]):
        p.grad = g
    state["at"] ^= 1
    opt.step()
    out = []
    for p in params:
        st = opt.state[p]
        one = [p.detach(), st["exp_avg"], st["exp_avg_sq"], st["exp_avg_diff"], st["prev_grad"]]
        if state["kind"] == "refresh":
            pre = st["preconditioner"]
            for leaf, _, _ in pre.leaves():
                one += ([leaf.L_ema_q, leaf.R_ema_q] if state["int8"]
                        else [leaf.L_ema, leaf.R_ema]) + [leaf.S_l, leaf.S_r]
        out.append(one)
    return out


# ----------------------------------------------------------------- exact ---

def _tikhonov_eig(a, bias, k, diagonal):
    a = a / bias
    a.diagonal().add_(max(1e-8, 1e-4 * float(a.trace()) / len(a)))
    if diagonal:
        w, order = a.diagonal().sort(stable=True)
        v = torch.eye(len(a), dtype=a.dtype, device=DEV)[:, order]
    else:
        w, v = torch.linalg.eigh(a)
    return w.flip(0).clamp(min=0.0)[:k], v.flip(1)[:, :k]


def _refresh64(case, blk, g):
    """A block's new EMAs, spectrum and eigenfactors."""
    bias = 1.0 - RHO ** (REFRESHES + 1)
    emas, outs, k = [], [], _rank(blk["m"], blk["n"], case["k"])
    for old, x in zip(blk["ema"], (g, g.T)):
        old = old[0].double() * old[1] if case["ema"] == "int8" else old.double()
        new = old * RHO + (1.0 - RHO) * (x @ x.T)
        if case["ema"] == "int8":
            q, scale = _codes(new)
            emas.append(None)
            new = q.double() * scale
        else:
            emas.append(new)
        outs.append(_tikhonov_eig(new, bias, k, case["spectrum"] == "diagonal"))
    return emas, [s for s, _ in outs], [u for _, u in outs]


def _step64(case, one):
    """What one SCAO.step leaves of a parameter, in 64 bits but for the
    places where the optimizer rounds to the parameter's type by definition."""
    dt = DTYPES[case["dtype"]]
    f64 = torch.float64

    def stored(x):
        return x.to(dt).double() if dt != torch.float32 else x

    m2, n2 = _flat(one["shape"])
    t = STEP + 1
    raw = one["grads"][0].reshape(m2, n2).to(f64)
    g = raw
    if case.get("sparsity", 0.0) > 0.0:
        ema = (FILTER_EMA * one["hist"].reshape(m2, n2).to(f64).abs()
               + (1.0 - FILTER_EMA) * raw.abs())
        flat = ema.reshape(-1).sort().values
        pos = case["sparsity"] * (len(flat) - 1)
        lo = int(math.floor(pos))
        hi = min(lo + 1, len(flat) - 1)
        thr = flat[lo] + (pos - lo) * (flat[hi] - flat[lo])
        g = raw * (ema >= thr)
    p = stored(one["p"].reshape(m2, n2).to(f64) * (1.0 - LR * WD))
    m, v, d = (one[n].reshape(m2, n2).to(f64) for n in ("exp_avg", "exp_avg_sq", "exp_avg_diff"))
    bc1, bc2, bc3 = (1.0 - b ** t for b in (BETA1, BETA2, BETA3))
    if case.get("phase") == 1:
        m = m * BETA1 + (1.0 - BETA1) * g
        v = v * BETA2 + (1.0 - BETA2) * g * g
        u = m / (v.sqrt() / math.sqrt(bc2) + EPS)
        p = stored(p - LR / bc1 * stored(u))
        return [p, m, v, d, g], []
    gp = torch.empty_like(raw)
    nat2, extra = 0.0, []
    for blk in one["blocks"]:
        rows, cols = slice(blk["r"], blk["r"] + blk["m"]), slice(blk["c"], blk["c"] + blk["n"])
        gb = raw[rows, cols]
        if not _kron(blk["m"], blk["n"]):
            h = one["hist"].reshape(m2, n2)[rows, cols].to(f64)
            ema, bias = (1.0 - RHO) * h * h, 1.0 - RHO
            if case["kind"] == "refresh":
                ema = ema * RHO + (1.0 - RHO) * gb * gb
                bias = 1.0 - RHO ** (REFRESHES + 1)
            gp[rows, cols] = gb / ((ema / bias).pow(0.25) + 1e-8)
            nat2 += float((gb * gb / (ema.sqrt() + EPS)).sum())
            continue
        if case["kind"] == "refresh":
            emas, s, u = _refresh64(case, blk, gb)
            extra += emas + s
        else:
            s, u = [x.double() for x in blk["S"]], [x.double() for x in blk["U"]]
        pr = u[0].T @ gb @ u[1]
        i4 = [x.clamp(min=1e-8).pow(-0.25) for x in s]
        i2 = [x.clamp(min=EPS).pow(-0.5) for x in s]
        gp[rows, cols] = gb + u[0] @ ((i4[0][:, None] * i4[1] - 1.0) * pr) @ u[1].T
        nat2 += float((i2[0][:, None] * pr * i2[1]).square().sum())
    gp, nat = stored(gp), math.sqrt(nat2)
    if nat > TAU:
        gp = stored(gp * (TAU / nat))
    diff = g - one["prev"].reshape(m2, n2).to(f64)
    m = m * BETA1 + (1.0 - BETA1) * gp
    d = d * BETA3 + (1.0 - BETA3) * diff
    gad = gp + (1.0 - BETA3) * diff
    v = v * BETA2 + (1.0 - BETA2) * gad * gad
    u = (m / bc1 + (1.0 - BETA3) * (d / bc3)) / ((v / bc2).sqrt() + EPS)
    pn, un = float(p.norm()), float(u.norm())
    trust = LARS * pn / (un + WD * pn + 1e-8) if pn and un else 1.0
    p = stored(p - LR * trust * stored(u))
    return [p, m, v, d, g], extra


def exact(case, seed):
    if case["kind"] in ("step", "refresh"):
        # which unit vectors a tied diagonal spectrum keeps is an order, not a number
        tied = case["kind"] == "refresh" and case["spectrum"] == "diagonal"
        out = []
        for one in _step_inputs(case, seed):
            five, extra = _step64(case, one)
            five = [x.reshape(one["shape"]) for x in five]
            if tied and len(one["shape"]) > 1:
                five = [None, None, None] + five[3:]
            out.append(five + extra)
        return out
    x = {n: v.double() if isinstance(v, torch.Tensor) else v
         for n, v in _matrix_inputs(case, seed).items()}
    if case["kind"] == "fused":
        p = x["U_l"].T @ x["G"] @ x["U_r"]
        return x["G"] + x["U_l"] @ ((x["s_l"][:, None] * x["s_r"] - 1.0) * p) @ x["U_r"].T
    return None, float((RHO * x["q"] * x["scale"] + x["v"]).abs().max()) / 127.0


# ------------------------------------------------------------------ work ---

def work(case):
    if case["kind"] == "fused":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=4 * (2 * m * n + (m + n) * k), flops=4 * m * n * k + 2 * (m + n) * k * k)
    if case["kind"] == "ema":
        return dict(bytes=6 * case["rows"] * case["cols"], flops=0)
    size = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    nbytes = flops = 0
    for shape in _shapes(case):
        m, n = _flat(shape)
        # parameter read and written, gradient read; four fp32 moments read
        # and written (Phase 1: two, and the last gradient written); the
        # filter's average read and written
        nbytes += m * n * (3 * size + (20 if case.get("phase") == 1 else 32)
                           + (8 if case.get("sparsity", 0.0) > 0 else 0))
        if case.get("phase") == 1:
            continue
        for bm, bn, _, _ in _blocks((m, n), case["dim"]):
            if not _kron(bm, bn):
                nbytes += 4 * bm * bn * (3 if case["kind"] == "refresh" else 1)
                continue
            k = _rank(bm, bn, case["k"])
            nbytes += 4 * (bm + bn) * (k + 1)
            flops += 4 * bm * bn * k + 2 * (bm + bn) * k * k
            if case["kind"] == "refresh":
                # Gram products (symmetric), the EMAs read and written, and
                # for dense ones reduction to tridiagonal form and k vectors
                flops += bm * bn * (bm + bn)
                nbytes += (2 if case["ema"] == "int8" else 8) * (bm * bm + bn * bn)
                if case["spectrum"] == "dense":
                    flops += sum(4 * d ** 3 // 3 + 2 * d * d * k for d in (bm, bn))
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # about four times what the path differs from exact() by, measured over
    # listed and drawn cases
    if case["kind"] == "fused":
        return {"rel": 4e-6, "max": 4e-5}
    if case["kind"] == "ema":
        return {"rel": 1e-6, "differ": 1e-5}
    if case["dtype"] != "fp32":
        # 16-bit parameters and preconditioned gradients: a value between two
        # neighbours of the type may round either way
        tol = {"rel": 1e-3, "max": 2e-2, "differ": 1e-4}
    elif case["kind"] == "refresh":
        # codes on the border of two values may fall on either side
        tol = {"rel": 2e-5, "max": 1e-2, "differ": 1e-4}
    else:
        tol = {"rel": 1e-6, "max": 1e-4}
    if case.get("sparsity", 0.0) > 0.0:
        # gradients whose average is on the threshold may be kept or dropped
        tol = {"rel": 1.2e-2, "max": 0.99}
    return tol
