"""The work that a user of this library has it do, as cases that can be timed:
likelihood evaluations of one fit (value and gradient), the Hessian of a fit
result, the normalisation integral that feeds them, the batched fits over bins
and starts, and the training of the learned start values.

Inputs are drawn with torch on the GPU from the seed alone, with the amplitude
recipe of the benchmark: A_i(e) = (N(0,1) + i N(0,1)) s_i exp(N(0,1)_e / 2) with
s_i ~ U[0.1, 1].  Data follow the model: an event's density is the pool's times
its intensity sigma(A) = sum_rs |sum_i T_rsi A_si|^2, sampled directly (a
component (r, s) by its share of the mean intensity, the amplitude's component
along it with a Gamma(2) square, the event scale's lognormal shifted), which is
what accept-rejected events are distributed as.
"""
import math

import numpy as np
import torch

from rootpwa_amd import batch as batch_mod
from rootpwa_amd import capi
from rootpwa_amd import likelihood as lik
from rootpwa_amd import mlp as mlp_mod

DEV = "cuda"
FDF, HESSIAN, INTEGRAL, BATCH, FIT, TRAIN = "fdf", "hessian", "integral", "batch", "fit", "train"


def listed():
    return [
        # the size of the reference's own GPU test, in Minuit's call pattern (value, then gradient)
        dict(name="fdf_10k", op=FDF, events=10_000, neg=7, pos=34, rank=2, mixed=False, minuit=True),
        # the small CPU-sized configuration of the benchmark: latency and launches count
        dict(name="fdf_100k", op=FDF, events=100_000, neg=0, pos=16, rank=1, mixed=False, minuit=False),
        # one mass bin of a binned fit, all waves in one sector, complex64 storage
        dict(name="fdf_bin", op=FDF, events=75_821, neg=0, pos=88, rank=1, mixed=True, minuit=False),
        # a ragged wave set at rank 3
        dict(name="fdf_rank3", op=FDF, events=300_007, neg=13, pos=40, rank=3, mixed=True, minuit=False),
        # the headline workload, both precisions
        dict(name="fdf_2M_fp64", op=FDF, events=2_000_000, neg=8, pos=80, rank=2, mixed=False, minuit=False),
        dict(name="fdf_2M_mixed", op=FDF, events=2_000_000, neg=8, pos=80, rank=2, mixed=True, minuit=False),
        # the errors of the headline fit's result
        dict(name="hessian_2M", op=HESSIAN, events=2_000_000, neg=8, pos=80, rank=2, mixed=True),
        # the headline's normalisation integral, and a weighted one of a small odd sample
        dict(name="integral_5M", op=INTEGRAL, events=5_000_000, waves=88, weighted=False),
        dict(name="integral_150k", op=INTEGRAL, events=150_001, waves=41, weighted=True),
        # one evaluation of all fits of the batched workload: 48 bins of 20k..400k events, 64 starts each
        dict(name="batch_48bins", op=BATCH, bins=48, low=20_000, high=400_000, waves=88, starts=64),
        # batched fits from start values near the minimum, as the learned initializer gives them, within a budget of
        # evaluations that most of them converge in (without one, the slowest fit's path alone would set the time)
        dict(name="fit_12bins", op=FIT, bins=12, low=20_000, high=100_000, waves=88, starts=8, budget=40),
        # five epochs of the initializer's network at the batch size it is trained with
        dict(name="train_1800", op=TRAIN, rows=1800, inputs=775, hidden=512, layers=3, outputs=176, batch=64, epochs=5),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice([FDF, FDF, FDF, FDF, HESSIAN, INTEGRAL, BATCH, FIT, TRAIN])
    if op == FDF:
        waves = _log(rng, 6, 88)
        neg = rng.choice([0, rng.randint(1, waves // 3)])
        return dict(op=op, events=_log(rng, 5_000, 2_000_000), neg=neg, pos=waves - neg, rank=rng.choice([1, 1, 2, 2, 3, 4]),
                    mixed=rng.random() < 0.5, minuit=rng.random() < 0.3)
    if op == HESSIAN:
        waves = _log(rng, 12, 88)
        neg = rng.choice([0, rng.randint(1, waves // 3)])
        return dict(op=op, events=_log(rng, 20_000, 1_000_000), neg=neg, pos=waves - neg, rank=rng.choice([1, 2]),
                    mixed=rng.random() < 0.5)
    if op == INTEGRAL:
        return dict(op=op, events=_log(rng, 50_000, 5_000_000), waves=_log(rng, 8, 88), weighted=rng.random() < 0.5)
    if op == BATCH:
        low = _log(rng, 5_000, 40_000)
        return dict(op=op, bins=_log(rng, 4, 48), low=low, high=low * 10, waves=_log(rng, 16, 88), starts=rng.randint(8, 64))
    if op == FIT:
        low = _log(rng, 10_000, 20_000)
        return dict(op=op, bins=rng.randint(3, 12), low=low, high=low * 5, waves=_log(rng, 16, 88), starts=rng.randint(1, 8), budget=40)
    waves, pairs = rng.randint(32, 88), rng.randint(64, 256)
    return dict(op=op, rows=rng.randint(400, 1800), inputs=3 * waves - 1 + 2 * pairs, hidden=rng.choice([128, 256, 512]),
                layers=rng.randint(1, 3), outputs=2 * waves, batch=rng.choice([32, 64, 64]), epochs=5)


# ---- inputs, from the seed alone ------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _cnormal(shape, g):
    """Complex normal values with unit variance of each part."""
    return torch.view_as_complex(torch.randn(tuple(shape) + (2,), dtype=torch.float64, device=DEV, generator=g))


def _scales(W, g):
    return 0.1 + 0.9 * torch.rand(W, dtype=torch.float64, device=DEV, generator=g)


def _pool(n, scales, g):
    """n events of the amplitude pool, [n][W]."""
    z = _cnormal((n, scales.numel()), g)
    z *= (torch.exp(0.5 * torch.randn((n, 1), dtype=torch.float64, device=DEV, generator=g)) * scales).to(z.dtype)
    return z


def _sums(scales, g, n=40_000):
    """Normalisation sums over a pool of n events."""
    a = _pool(n, scales, g)
    return a.T @ a.conj(), n


def _data(n, scales, T, nW, g):
    """n events distributed as the pool's times sigma under T [rank][W] (refl -1 waves first)."""
    W = scales.numel()
    z = _cnormal((n, W), g)
    parts = []
    for r in range(T.shape[0]):
        for off, w in ((0, nW[0]), (nW[0], nW[1])):
            if w and float(T[r, off:off + w].abs().sum()) > 0:
                t = torch.zeros(W, dtype=torch.complex128, device=DEV)
                t[off:off + w] = T[r, off:off + w] * scales[off:off + w]
                parts.append(t)
    t = torch.stack(parts)
    share = (t.abs() ** 2).sum(1)
    which = torch.multinomial(share / share.sum(), n, replacement=True, generator=g)
    t = t / torch.sqrt(share)[:, None]
    u = torch.rand((2, n), dtype=torch.float64, device=DEV, generator=g).clamp_(1e-300)
    size = torch.sqrt(-2.0 * torch.log(u[0] * u[1]))  # |c|^2 / 2 ~ Gamma(2)
    for k in range(t.shape[0]):
        at = torch.nonzero(which == k).flatten()
        zk = z[at]
        c = zk @ t[k]
        zk += ((c / c.abs()) * size[at] - c)[:, None] * t[k].conj()[None, :]
        z[at] = zk
    z *= (torch.exp(0.5 * (1.0 + torch.randn((n, 1), dtype=torch.float64, device=DEV, generator=g))) * scales).to(z.dtype)
    return z


def _restrict(T, nW):
    """The rank restrictions of the likelihood: 0 for wave < rank, real for wave = rank of a sector."""
    for r in range(T.shape[0]):
        for off, w in ((0, nW[0]), (nW[0], nW[1])):
            T[r, off:off + min(r, w)] = 0
            if r < w:
                T[r, off + r] = T[r, off + r].abs().to(T.dtype)
    return T


def _fit_inputs(case, seed):
    """Data, sums and a point of a single fit: T [rank][W] of normalised amplitudes near the minimum's size, and the flat wave."""
    g = _gen(seed)
    nW = (case["neg"], case["pos"])
    W, rank, N = sum(nW), case["rank"], case["events"]
    scales = _scales(W, g)
    sums, M = _sums(scales, g)
    truth = _restrict(_cnormal((rank, W), g), nW)
    amps = _data(N, scales, truth, nW, g)
    T = _restrict(truth * scales + 0.2 * _cnormal((rank, W), g), nW)
    T = T * math.sqrt(N) / float(torch.sqrt((T.abs() ** 2).sum()))
    return amps, sums, M, T, 0.1 * math.sqrt(N / (1.0 + W))


def _par(T, flat, nW):
    """The likelihood's parameter vector: rank, sector, wave; real anchors; the flat wave last."""
    T = T.cpu().numpy()
    par = []
    for r in range(T.shape[0]):
        for off, w in ((0, nW[0]), (nW[0], nW[1])):
            for i in range(r, w):
                par.append(T[r, off + i].real)
                if i > r:
                    par.append(T[r, off + i].imag)
    return np.array(par + [flat])


def _par_slots(rank, nW):
    """(rank, wave, 0 real / 1 imaginary) of every parameter but the flat one."""
    out = []
    for r in range(rank):
        for off, w in ((0, nW[0]), (nW[0], nW[1])):
            for i in range(r, w):
                out.append((r, off + i, 0))
                if i > r:
                    out.append((r, off + i, 1))
    return out


def _bin_sizes(case, seed):
    rng = np.random.default_rng(seed + 5)
    return np.exp(rng.uniform(math.log(case["low"]), math.log(case["high"]), case["bins"])).astype(np.int64)


def _bins(case, seed):
    """Per bin: data, sums, the pool's size, and the true T of normalised amplitudes at the minimum's size, real at wave 0."""
    g = _gen(seed)
    W = case["waves"]
    for n in _bin_sizes(case, seed):
        scales = _scales(W, g)
        sums, M = _sums(scales, g)
        truth = _cnormal((1, W), g)
        amps = _data(int(n), scales, truth, (0, W), g)
        T = truth[0] * scales * (truth[0, 0].abs() / truth[0, 0])
        yield amps, sums, M, T * math.sqrt(int(n)) / float(torch.sqrt((T.abs() ** 2).sum()))


def _batch_par(T, flat):
    """T [starts][W] with a real wave 0 -> [starts][2 W]."""
    p = np.zeros((T.shape[0], 2 * T.shape[1]))
    p[:, 0] = T[:, 0].real
    p[:, 1:-1:2] = T[:, 1:].real
    p[:, 2:-1:2] = T[:, 1:].imag
    p[:, -1] = flat
    return p


def _starts(case, seed):
    """Points [bins][starts][2 W] of an evaluation, as the fits' random starts are drawn: uniform size up to sqrt(N), random
    sign."""
    rng = np.random.default_rng(seed + 6)
    W, S = case["waves"], case["starts"]
    out = []
    for n in _bin_sizes(case, seed):
        p = rng.uniform(0.01, math.sqrt(n), (S, 2 * W)) * np.where(rng.random((S, 2 * W)) < 0.5, -1.0, 1.0)
        out.append(p)
    return np.array(out)


def _near(T, n, S, rng):
    """Start values [S][2 W] of a fit, some per cent off the true point."""
    T = T.cpu().numpy()
    size = np.sqrt(np.mean(np.abs(T) ** 2))
    t = T[None, :] + 0.05 * size / math.sqrt(2) * (rng.standard_normal((S, T.size)) + 1j * rng.standard_normal((S, T.size)))
    t[:, 0] = np.abs(t[:, 0])
    return _batch_par(t, 0.02 * math.sqrt(n))


def _network_inputs(case, seed):
    """Standardised features, and targets that depend on them, as the initializer trains on."""
    rng = np.random.default_rng(seed + 7)
    X = rng.standard_normal((case["rows"], case["inputs"])).astype(np.float32)
    mix = rng.standard_normal((case["inputs"], case["outputs"])) / math.sqrt(case["inputs"])
    T = np.tanh(X @ mix) + 0.5 * rng.standard_normal((case["rows"], case["outputs"]))
    dims = [case["inputs"]] + [case["hidden"]] * case["layers"] + [case["outputs"]]
    p = []
    for a, b in zip(dims[:-1], dims[1:]):
        lim = math.sqrt(6.0 / (a + b))
        p += [rng.uniform(-lim, lim, a * b), np.zeros(b)]
    return X, T.astype(np.float32), np.concatenate(p).astype(np.float32), dims


# ---- what a program has in hand before the call ----------------------------------

def _likelihood(case, amps, sums, M):
    nW = (case["neg"], case["pos"])
    waves = [("n%03d" % i, -1, 0.0) for i in range(nW[0])] + [("p%03d" % i, 1, 0.0) for i in range(nW[1])]
    names = [w[0] for w in waves]
    L = lik.pwaLikelihood(capi.PREC_MIXED if case["mixed"] else capi.PREC_FP64)
    L.init(waves, case["rank"])
    m = lik.ampIntegralMatrix(names)
    m.setSums(sums.cpu().numpy(), M)
    L.addNormIntegral(m)
    L.addAccIntegral(m)
    torch.cuda.synchronize()
    L.addAmplitudesDevice(amps.data_ptr(), case["events"])
    L.finishInit()
    return L


def prepare(case, seed):
    op = case["op"]
    if op in (FDF, HESSIAN):
        lik.pwaLikelihood.setQuiet(True)
        amps, sums, M, T, flat = _fit_inputs(case, seed)
        L = _likelihood(case, amps, sums, M)
        return dict(op=op, L=L, par=_par(T, flat, (case["neg"], case["pos"])), minuit=case.get("minuit", False))
    if op == INTEGRAL:
        g = _gen(seed)
        a = _pool(case["events"], _scales(case["waves"], g), g)
        w = 0.5 + torch.rand(case["events"], dtype=torch.float64, device=DEV, generator=g) if case["weighted"] else None
        torch.cuda.synchronize()
        return dict(op=op, amps=a, weights=w, M=case["events"], W=case["waves"])
    if op in (BATCH, FIT):
        B = batch_mod.BatchFit(case["waves"], case["starts"])
        rng = np.random.default_rng(seed + 8)
        near = []
        for amps, sums, M, T in _bins(case, seed):
            torch.cuda.synchronize()
            B.addBinDevice(amps.data_ptr(), amps.shape[0], sums.cpu().numpy(), M)
            near.append(_near(T, amps.shape[0], case["starts"], rng))
        B.finish()
        return dict(op=op, B=B, par=_starts(case, seed) if op == BATCH else np.array(near), budget=case.get("budget"))
    X, T, p, dims = _network_inputs(case, seed)
    net = mlp_mod.MLP(dims[0], case["hidden"], case["layers"], dims[-1], seed=1)
    return dict(op=op, net=net, X=X, T=T, p=p, batch=case["batch"], epochs=case["epochs"])


# ---- one pass --------------------------------------------------------------------

def run(s):
    op = s["op"]
    if op == FDF:
        if s["minuit"]:
            return np.float64(s["L"].DoEval(s["par"])), s["L"].Gradient(s["par"])
        value, gradient = s["L"].FdF(s["par"])
        return np.float64(value), gradient
    if op == HESSIAN:
        return s["L"].Hessian(s["par"])
    if op == INTEGRAL:
        return capi.integral_device(s["amps"].data_ptr(), s["M"], s["W"], None if s["weights"] is None else s["weights"].data_ptr())
    if op == BATCH:
        return s["B"].eval(s["par"])
    if op == FIT:
        par, value, _, _ = s["B"].fit(s["par"], maxEvaluations=s["budget"])
        return par, value
    s["net"].setParams(s["p"])
    loss = s["net"].train(s["X"], s["T"], batchSize=s["batch"], epochs=s["epochs"], lr=1e-4, seed=3)
    return loss, s["net"].params()


def work(case):
    op = case["op"]
    if op in (FDF, HESSIAN):
        N, W, R = case["events"], case["neg"] + case["pos"], case["rank"]
        size = N * W * (8 if case["mixed"] else 16)
        if op == FDF:
            return dict(bytes=size + 16 * 2 * R * W, flops=16 * N * W * R)
        D = 2 * R * W + 1
        return dict(bytes=size + 8 * D * D, flops=N * (D * (D + 1) + 4 * (case["neg"] ** 2 + case["pos"] ** 2) + 8 * W * R))
    if op == INTEGRAL:
        M, W = case["events"], case["waves"]
        return dict(bytes=16 * M * W + (8 * M if case["weighted"] else 0) + 16 * W * W, flops=4 * M * W * (W + 1))
    if op in (BATCH, FIT):
        # the mean of the log-uniform sizes; a fit from near the minimum takes about 30 evaluations
        n = case["bins"] * (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
        W, S = case["waves"], case["starts"]
        evals = 30 if op == FIT else 1
        return dict(bytes=evals * (n * W * 8 + 2 * case["bins"] * S * 2 * W * 8), flops=evals * 16 * n * W * S)
    dims = [case["inputs"]] + [case["hidden"]] * case["layers"] + [case["outputs"]]
    n = sum((a + 1) * b for a, b in zip(dims[:-1], dims[1:]))
    steps = case["epochs"] * (case["rows"] // min(case["batch"], case["rows"]))
    # parameters, gradient-free Adam state read and written each step; forward and both backward products
    return dict(bytes=steps * 24 * n, flops=steps * 6 * n * min(case["batch"], case["rows"]))


def tolerance(case):
    """About four times the largest error against exact() seen over the ranges (two seeds each); a fit's from paths whose
    start values differ in the last single-precision bit, budget and all."""
    op = case["op"]
    if op == FDF:
        return dict(rel=8e-7, max=3e-6) if case["mixed"] else dict(rel=2e-13, max=1e-12)
    if op == HESSIAN:
        return dict(rel=4e-8, max=2e-7) if case["mixed"] else dict(rel=1e-13, max=2e-12)
    if op == INTEGRAL:
        return dict(rel=6e-14, max=2e-13)
    if op == BATCH:
        return dict(rel=2e-7, max=1e-6)
    if op == FIT:
        return dict(rel=3e-2, max=0.9)
    return dict(rel=2e-6, max=6e-4)


# ---- the same in 64 bits, with torch alone ----------------------------------------

CHUNK = 100_000


def _normalised(amps, sums, M):
    d = torch.sqrt(torch.real(torch.diag(sums)) / M)
    amps /= d.to(amps.dtype)
    return amps, (sums / M) / (d[:, None] * d[None, :])


def _sectors(nW):
    return [(off, off + w) for off, w in ((0, nW[0]), (nW[0], nW[1])) if w]


def exact(case, seed):
    op = case["op"]
    if op in (FDF, HESSIAN):
        nW = (case["neg"], case["pos"])
        rank = case["rank"]
        amps, sums, M, T, flat = _fit_inputs(case, seed)
        amps, I = _normalised(amps, sums, M)
        return _exact_fdf(amps, I, T, flat, nW) if op == FDF else _exact_hessian(amps, I, T, flat, nW, rank)
    if op == INTEGRAL:
        g = _gen(seed)
        a = _pool(case["events"], _scales(case["waves"], g), g)
        w = 1.0 / (0.5 + torch.rand(case["events"], dtype=torch.float64, device=DEV, generator=g)) if case["weighted"] else None
        out = torch.zeros((case["waves"],) * 2, dtype=torch.complex128, device=DEV)
        for k in range(0, case["events"], CHUNK):
            x = a[k:k + CHUNK]
            out += (x if w is None else x * w[k:k + CHUNK, None]).T @ x.conj()
        if w is not None:
            out *= case["events"] / float(w.sum())
        return out.cpu().numpy()
    if op == BATCH:
        par = _starts(case, seed)
        value, grad = np.zeros(par.shape[:2]), np.zeros_like(par)
        for b, (amps, sums, M, _) in enumerate(_bins(case, seed)):
            amps, I = _normalised(amps, sums, M)
            value[b], grad[b] = _exact_starts(amps, I, torch.from_numpy(par[b]).to(DEV))
        return value, grad
    if op == TRAIN:
        return _exact_train(case, seed)
    return None  # a fit's path has no 64-bit counterpart


def _exact_fdf(amps, I, T, flat, nW):
    rank, W = T.shape
    value, dflat = 0.0, 0.0
    dT = torch.zeros_like(T)
    for k in range(0, amps.shape[0], CHUNK):
        x = amps[k:k + CHUNK]
        S = {(r, a): x[:, a:b] @ T[r, a:b] for r in range(rank) for a, b in _sectors(nW)}
        sigma = sum(v.abs() ** 2 for v in S.values()) + flat * flat
        value -= float(torch.log(sigma).sum())
        dflat -= 2 * flat * float((1 / sigma).sum())
        for r in range(rank):
            for a, b in _sectors(nW):
                dT[r, a:b] -= 2 * ((S[r, a] / sigma) @ x[:, a:b].conj())
    for r in range(rank):
        for a, b in _sectors(nW):
            u = I[a:b, a:b].conj() @ T[r, a:b]
            value += float(torch.real(torch.dot(T[r, a:b].conj(), u)))
            dT[r, a:b] += 2 * u
    value += flat * flat
    dflat += 2 * flat
    return np.float64(value), _par(dT, dflat, nW)


def _exact_hessian(amps, I, T, flat, nW, rank):
    slots = _par_slots(rank, nW)
    D = len(slots) + 1
    r_ = torch.tensor([s[0] for s in slots], device=DEV)
    w_ = torch.tensor([s[1] for s in slots], device=DEV)
    im = torch.tensor([s[2] for s in slots], device=DEV)
    sec = (w_ >= nW[0]).long()
    H = torch.zeros((D, D), dtype=torch.float64, device=DEV)
    W = sum(nW)
    Q = torch.zeros((W, W), dtype=torch.complex128, device=DEV)  # sum 2 / sigma a_i conj(a_j)
    for k in range(0, amps.shape[0], CHUNK):
        x = amps[k:k + CHUNK]
        S = torch.zeros((x.shape[0], rank, 2), dtype=torch.complex128, device=DEV)
        for r in range(rank):
            S[:, r, 0] = x[:, :nW[0]] @ T[r, :nW[0]] if nW[0] else 0
            S[:, r, 1] = x[:, nW[0]:] @ T[r, nW[0]:] if nW[1] else 0
        sigma = (S.abs() ** 2).sum((1, 2)) + flat * flat
        v = torch.empty((x.shape[0], D), dtype=torch.float64, device=DEV)
        d = S[:, r_, sec] * x[:, w_].conj()
        v[:, :-1] = torch.where(im[None, :] == 1, d.imag, d.real)
        v[:, -1] = flat
        v *= (2 / sigma)[:, None]
        H += v.T @ v
        y = x * torch.sqrt(2 / sigma)[:, None]
        Q += y.T @ y.conj()
        H[-1, -1] -= (2 / sigma).sum()
    B = 2 * I - Q
    b = B[w_][:, w_]
    same = (r_[:, None] == r_[None, :]) & (sec[:, None] == sec[None, :])
    term = torch.where(im[:, None] == im[None, :], b.real, torch.where(im[None, :] == 1, b.imag, -b.imag))
    H[:-1, :-1] += torch.where(same, term, torch.zeros_like(term))
    H[-1, -1] += 2
    return H.cpu().numpy()


def _exact_starts(amps, I, par):
    """Value and gradient of one bin at [starts][2 W]."""
    W = amps.shape[1]
    re, im = torch.zeros((par.shape[0], W), dtype=torch.float64, device=DEV), torch.zeros((par.shape[0], W), dtype=torch.float64, device=DEV)
    re[:, 0], re[:, 1:], im[:, 1:] = par[:, 0], par[:, 1:-1:2], par[:, 2:-1:2]
    T = torch.complex(re, im)
    flat2 = par[:, -1] ** 2
    value = torch.zeros(par.shape[0], dtype=torch.float64, device=DEV)
    inv = torch.zeros_like(value)
    dT = torch.zeros_like(T)
    for k in range(0, amps.shape[0], CHUNK):
        x = amps[k:k + CHUNK]
        S = x @ T.T.contiguous()
        sigma = S.abs() ** 2 + flat2
        value -= torch.log(sigma).sum(0)
        inv += (1 / sigma).sum(0)
        dT -= 2 * ((S / sigma).T.contiguous() @ x.conj())
    u = T @ I.conj().T.contiguous()
    value += torch.real((T.conj() * u).sum(1)) + flat2
    dT += 2 * u
    g = torch.zeros_like(par)
    g[:, 0], g[:, 1:-1:2], g[:, 2:-1:2] = dT[:, 0].real, dT[:, 1:].real, dT[:, 1:].imag
    g[:, -1] = 2 * par[:, -1] * (1 - inv)
    return value.cpu().numpy(), g.cpu().numpy()


def _mix64(x):
    """The 64-bit mixing function that the documented shuffle of the training rows is drawn with."""
    m = (1 << 64) - 1
    x = (x + 0x9E3779B97F4A7C15) & m
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & m
    return x ^ (x >> 31)


def _exact_train(case, seed):
    X, T, p, dims = _network_inputs(case, seed)
    X, T, p = (torch.from_numpy(v.astype(np.float64)).to(DEV) for v in (X, T, p))
    n, B, steps = case["rows"], min(case["batch"], case["rows"]), 0
    m1, m2 = torch.zeros_like(p), torch.zeros_like(p)
    losses = []
    for epoch in range(case["epochs"]):
        perm = list(range(n))
        for i in range(n - 1, 0, -1):
            j = _mix64(3 ^ _mix64(((epoch << 32) + i) & ((1 << 64) - 1))) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        perm = torch.tensor(perm, device=DEV)
        total = 0.0
        for k in range(n // B):
            at = perm[k * B:(k + 1) * B]
            q = p.clone().requires_grad_(True)
            h, off = X[at], 0
            for a, (i, o) in enumerate(zip(dims[:-1], dims[1:])):
                h = h @ q[off:off + i * o].view(i, o) + q[off + i * o:off + (i + 1) * o]
                off += (i + 1) * o
                if a + 2 < len(dims):
                    h = torch.nn.functional.gelu(h)
            loss = ((h - T[at]) ** 2).mean()
            g, = torch.autograd.grad(loss, q)
            total += float(loss.detach())
            steps += 1
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            p = p - 1e-4 * (m1 / (1 - 0.9 ** steps)) / (torch.sqrt(m2 / (1 - 0.999 ** steps)) + 1e-8)
        losses.append(total / (n // B))
    return np.array(losses, dtype=np.float64), p.cpu().numpy()
