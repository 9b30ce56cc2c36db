"""Performance cases of the Brownian-dynamics framework.

Each case is one call, or one short program of calls, that a user of the
package makes through its public entry points:

  traj      a stretch of trajectory: start state in, k predictor-corrector
            steps, state and energies out (BDEngine)
  forces    one force pass with the forces and the energy on the host, as for
            an energy analysis of a frame (BDEngine.forces)
  cholesky  the factor of a caller's matrix in device memory (bd_cholesky)
  pairs     the core-core charge term and its adjoint (CoreCorePairs)
  gradient  loss and parameter gradients of a short trajectory (DiffBD)

Sizes are those of the package's own configurations (12, 50, 100, 500 and
1000 nucleosomes; 5 tails of 10 beads and 300 charges per core; 22 free
linker-histone beads where bound), and odd ones between them.
"""
import ctypes
import math

import numpy as np
import torch

from brownian_dynamics_cuda_amd import diff as Df
from brownian_dynamics_cuda_amd import engine as E
from brownian_dynamics_cuda_amd import fiber as Fb
from brownian_dynamics_cuda_amd import system as S

MODES = {"fp64": E.CHOL_FP64, "fp32": E.CHOL_FP32, "bf16": E.CHOL_BF16}


def listed():
    return [
        # the smallest fiber in daily use, one host call per step: the noise goes up and the
        # energy comes back at each step, so latency and launches count
        traj("step_12", 12, lh=False, feed="step", steps=20),
        # a deck as the host driver runs it by default: linker histones bound, all beads
        # (tails and linker histones too) in the hydrodynamic tensor, D of 2826 rows
        traj("deck_12_all_beads", 12, lh=True, hi_all=True, feed="batch", steps=10),
        # a mid-sized fiber in batches of host noise, as the driver feeds it between samples
        traj("batch_50", 50, lh=False, feed="batch", steps=20),
        # the headline fiber, noise resident in device memory
        traj("device_100", 100, lh=True, feed="device", steps=20),
        # an odd size between the configurations, FP32 trailing updates with the FP64 refinement
        traj("batch_157_fp32", 157, lh=True, feed="batch", steps=8, mode="fp32"),
        # a large fiber without linker histones, everything FP64
        traj("batch_500", 500, lh=False, feed="batch", steps=2),
        # the largest fiber, with linker histones, in FP64 and with BF16 trailing updates
        traj("batch_1000", 1000, lh=True, feed="batch", steps=1),
        traj("batch_1000_bf16", 1000, lh=True, feed="batch", steps=2, mode="bf16"),
        # energy and forces of a frame, read back to the host
        dict(name="forces_300", kind="forces", n_c=300, lh=True, linkers=6),
        # a host program's own tensor, factored in device memory; a ragged size
        dict(name="cholesky_3001", kind="cholesky", m=3001),
        # the differentiable form's pair term in its default arithmetic, forward and backward
        dict(name="pairs_50_f32", kind="pairs", n_c=50, linkers=6, dtype="float32"),
        # the differentiable trajectory, forward and backward, with FP64 forces
        dict(name="gradient_50", kind="gradient", n_c=50, linkers=6, steps=2, loss="end_to_end"),
    ]


def traj(name, n_c, lh, feed, steps, mode="fp64", hi_all=False, linkers=6):
    return dict(name=name, kind="traj", n_c=n_c, lh=lh, hi_all=hi_all, linkers=linkers, mode=mode,
                feed=feed, steps=steps)


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["traj", "traj", "traj", "all", "forces", "cholesky", "pairs", "gradient"])
    linkers = rng.choice([5, 6, 6, 7])
    if kind == "traj":
        n_c = log_int(rng, 10, 850)
        c = traj("", n_c, rng.random() < 0.5, rng.choice(["step", "batch", "device"]), 1,
                 rng.choice(["fp64", "fp64", "fp32", "bf16"]), False, linkers)
        c["steps"] = max(1, min(20, 600 // n_c)) if n_c < 300 else 1
    elif kind == "all":
        n_c = log_int(rng, 4, 32)
        c = traj("", n_c, rng.random() < 0.5, rng.choice(["step", "batch"]), max(1, 100 // n_c),
                 "fp64", True, linkers)
    elif kind == "forces":
        c = dict(kind="forces", n_c=log_int(rng, 10, 1000), lh=rng.random() < 0.5, linkers=linkers)
    elif kind == "cholesky":
        c = dict(kind="cholesky", m=log_int(rng, 150, 9000))
    elif kind == "pairs":
        c = dict(kind="pairs", n_c=log_int(rng, 10, 500), linkers=linkers,
                 dtype=rng.choice(["float32", "float64"]))
    else:
        loss = rng.choice(["end_to_end", "energy"])  # the energy takes one more force pass
        c = dict(kind="gradient", n_c=log_int(rng, 10, 50), linkers=linkers,
                 steps=1 if loss == "energy" else rng.choice([1, 2]), loss=loss)
    c.pop("name", None)
    return c


def fiber(case, seed):
    """A generated fiber with thermal displacements, so that its linkers are
    not straight and no two of its bonds are alike."""
    fib, st = Fb.make_fiber(case["n_c"], seed=seed, with_lh=case.get("lh", False),
                            linker_beads=case["linkers"], hi_all=int(case.get("hi_all", False)))
    rng = np.random.default_rng(seed + 1)
    moved = [x + 0.05 * rng.standard_normal(x.size) for x in (st.r, st.r_t, st.r_lh)]
    return fib, S.State(moved[0], st.a, st.b, st.c, moved[1], moved[2])


def noise(fib, steps, seed):
    g = E.HostRng(seed % (1 << 31))
    n_D3 = 3 * (fib.n + fib.n_tail + fib.n_LH)
    drawn = [g.step_noise(k, fib.r_var(), n_D3) for k in range(steps)]
    return np.stack([d[0] for d in drawn]), np.stack([d[1] for d in drawn])


def tensor_of_beads(m, seed):
    """Rotne-Prager-Yamakawa tensor of a chain of beads of 1.5 nm radius, its
    first m rows and columns, on the GPU."""
    n = m // 3 + 1
    g = torch.Generator().manual_seed(seed)
    way = torch.randn(n, 3, generator=g, dtype=torch.float64)
    x = torch.cumsum(3.1 * way / way.norm(dim=1, keepdim=True), 0).cuda()
    rad = 1.5
    z = x[:, None, :] - x[None, :, :]
    s = z.norm(dim=2) + torch.eye(n, dtype=torch.float64, device="cuda")
    far = s >= 2 * rad
    c0 = torch.where(far, 0.75 * rad / s * (1 + 2 * rad ** 2 / (3 * s * s)), 1 - 9 * s / (32 * rad))
    c1 = torch.where(far, 0.75 * rad / s * (1 - 2 * rad ** 2 / (s * s)), 3 * s / (32 * rad))
    own = torch.eye(n, dtype=torch.bool, device="cuda")
    c0 = c0.masked_fill(own, 1.0)
    c1 = c1.masked_fill(own, 0.0)
    D = torch.empty(n, 3, n, 3, dtype=torch.float64, device="cuda")
    for k in range(3):
        for j in range(3):
            D[:, k, :, j] = c1 * z[..., k] * z[..., j] / (s * s) + (c0 if k == j else 0.0)
    return D.reshape(3 * n, 3 * n)[:m, :m].contiguous()


def pair_inputs(case, seed):
    """Charge sites, charges, partner lists and the cotangents of the pair term."""
    fib, st = fiber(case, seed)
    dt = getattr(torch, case["dtype"])
    cores = np.nonzero(fib.types == 1)[0]
    r, a, b, c = (x.reshape(-1, 3)[cores] for x in (st.r, st.a, st.b, st.c))
    p = np.asarray(fib.core_pos).reshape(-1, 3)
    Q = (r[:, None] + a[:, None] * p[None, :, :1] + b[:, None] * p[None, :, 1:2]
         + c[:, None] * p[None, :, 2:])
    near = np.linalg.norm(r[:, None] - r[None], axis=2) <= 25.0
    np.fill_diagonal(near, False)
    off = np.concatenate([[0], np.cumsum(near.sum(1))]).astype(np.int32)
    nbr = np.nonzero(near)[1].astype(np.int32)
    rng = np.random.default_rng(seed + 2)
    gpu = [torch.tensor(np.ascontiguousarray(x), device="cuda") for x in
           (Q, fib.core_q, off, nbr, rng.standard_normal(Q.shape), rng.standard_normal(len(cores)))]
    ph = fib.phys
    return dict(Q=gpu[0].to(dt), q=gpu[1].to(dt), off=gpu[2], nbr=gpu[3], gf=gpu[4].to(dt),
                ge=gpu[5].to(dt), consts=(ph.k_e, ph.debye, ph.k_ex, ph.sig_cc))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "cholesky":
        D = tensor_of_beads(case["m"], seed)
        return dict(kind=kind, m=case["m"], D=D, lib=E.load_library())
    if kind == "pairs":
        return dict(kind=kind, **pair_inputs(case, seed))
    fib, st = fiber(case, seed)
    if kind == "gradient":
        rr, p = noise(fib, case["steps"], seed)
        return dict(kind=kind, bd=Df.DiffBD(fib, force_dtype=torch.float64), st=st, rr=rr, p=p,
                    loss=case["loss"])
    eng = E.BDEngine(fib, chol_mode=MODES[case.get("mode", "fp64")])
    eng.set_state(st)
    if kind == "forces":
        return dict(kind=kind, eng=eng, st=st)
    rr, p = noise(fib, case["steps"], seed)
    state = dict(kind=kind, eng=eng, st=st, rr=rr, p=p, feed=case["feed"])
    if case["feed"] == "device":
        state["d_rr"], state["d_p"] = torch.tensor(rr, device="cuda"), torch.tensor(p, device="cuda")
        state["d_e"] = torch.zeros(len(rr), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
    return state


def run(state):
    kind = state["kind"]
    if kind == "traj":
        eng, rr, p = state["eng"], state["rr"], state["p"]
        eng.set_state(state["st"])
        if state["feed"] == "batch":
            energy = eng.run_steps(rr, p)
        elif state["feed"] == "step":
            energy = np.array([eng.step(rr[k], p[k]) for k in range(len(rr))])
        else:
            d_rr, d_p, energy = state["d_rr"], state["d_p"], state["d_e"]
            for k in range(len(rr)):
                eng.step_device(d_rr[k].data_ptr(), d_p[k].data_ptr(), energy[k].data_ptr())
        out = eng.get_state()
        return dict(energy=energy, r=out.r, a=out.a, b=out.b, c=out.c, r_t=out.r_t, r_lh=out.r_lh)
    if kind == "forces":
        state["eng"].set_state(state["st"])
        return state["eng"].forces()
    if kind == "cholesky":
        lib, m, D = state["lib"], state["m"], state["D"]
        L = torch.empty_like(D)
        neg = ctypes.c_int(0)
        stream = torch.cuda.current_stream().cuda_stream
        if lib.bd_cholesky(m, D.data_ptr(), m, L.data_ptr(), m, E.CHOL_FP64, ctypes.byref(neg), stream):
            raise E.BDError(lib.bd_last_error().decode())
        return dict(L=L, neg=neg.value)
    if kind == "pairs":
        Q = state["Q"].detach().requires_grad_(True)
        q = state["q"].detach().requires_grad_(True)
        f, e = Df.CoreCorePairs.apply(Q, q, state["off"], state["nbr"], state["consts"])
        gQ, gq = torch.autograd.grad((f, e), (Q, q), (state["gf"], state["ge"]))
        return dict(f=f, e=e, gQ=gQ, gq=gq)
    loss, grads = state["bd"].gradients(state["st"], state["rr"], state["p"], loss=state["loss"])
    return dict(loss=loss, **grads)


def exact(case, seed):
    if case["kind"] == "cholesky":
        return dict(L=torch.linalg.cholesky(tensor_of_beads(case["m"], seed)), neg=0)
    if case["kind"] == "pairs":
        return exact_pairs(**pair_inputs(case, seed))
    return None  # a whole step or force pass: no plain form of it in a few lines


def exact_pairs(Q, q, off, nbr, gf, ge, consts):
    ke, kappa, kex, sigma = consts
    Q = Q.double().requires_grad_(True)
    q = q.double().requires_grad_(True)
    off, nbr = off.cpu().tolist(), nbr.cpu().tolist()
    fs, es = [], []
    for i in range(len(Q)):
        js = nbr[off[i]:off[i + 1]]
        z = Q[i][:, None, :] - Q[js].reshape(1, -1, 3)
        d = z.norm(dim=2)
        qq = ke * q[:, None] * q.repeat(len(js))[None, :]
        dh = torch.exp(-kappa * d) * qq
        sd6 = (sigma / d) ** 6
        ev = d <= 8.0
        g = dh * (kappa * d + 1) / (d * d) + torch.where(ev, kex * (12 * sd6 * sd6 - 6 * sd6) / d, 0.0 * d)
        u = dh / d + torch.where(ev, kex * (sd6 * sd6 - sd6), 0.0 * d)
        fs.append(((g / d)[..., None] * z).sum(1))
        es.append(0.5 * u.sum())
    f, e = torch.stack(fs), torch.stack(es)
    gQ, gq = torch.autograd.grad((f, e), (Q, q), (gf.double(), ge.double()))
    return dict(f=f.detach(), e=e.detach(), gQ=gQ, gq=gq)


def work(case):
    """Bytes and operations one pass cannot do without: each input read and each
    output written once, the factor's m^3 / 3, and 38 operations for each
    charge pair of core pairs within 25 nm (about 5.7 pairs of cores per
    core)."""
    if case["kind"] == "cholesky":
        m = case["m"]
        return dict(bytes=8 * (m * (m + 1) // 2 + m * m), flops=m ** 3 / 3)
    n_c = case["n_c"]
    pairs = min(5.7 * n_c, n_c * (n_c - 1) / 2) * 300 * 300
    if case["kind"] == "pairs":
        w = 4 if case["dtype"] == "float32" else 8
        return dict(bytes=w * n_c * 300 * 3 * 4, flops=(38 + 80) * pairs)
    n = n_c + (n_c - 1) * case["linkers"]
    beads = n + 50 * n_c + (22 * n_c if case.get("lh") else 0)
    state = 8 * (12 * n + 3 * (beads - n))
    if case["kind"] == "forces":
        return dict(bytes=state + 8 * (6 * n + 3 * (beads - n)), flops=38 * pairs)
    m = 3 * (beads if case.get("hi_all") else n)
    k = case["steps"]
    if case["kind"] == "gradient":
        return dict(bytes=k * 8 * (6 * n + 3 * beads), flops=k * (m ** 3 + 4 * (38 + 80) * pairs))
    return dict(bytes=2 * state + k * 8 * (3 * n + 3 * beads),
                flops=k * (m ** 3 / 3 + 2 * 38 * pairs))
