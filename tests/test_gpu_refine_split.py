"""Batched refinement at the edges of its work split: windows whose samples end
just before, at and after a segment (1024 samples), whose channels end around
a chunk (32 for these windows alone, 256 for a plan of many), and scans whose
points end around a pass (3 points)."""
import numpy as np
import pytest

import frac_ddtr_ref as ref

pytestmark = pytest.mark.gpu

# (channels, samples)
WINDOWS = [(1, 1), (3, 4), (255, 255), (256, 256), (257, 257), (64, 1023), (300, 1024), (70, 1025), (512, 2048),
           (513, 2049), (33, 4095), (260, 4096)]


def _windows(cuda, seed):
    import torch
    g = torch.Generator(device=cuda).manual_seed(seed)
    off, ds_off, tables, xs = [], [], [], []
    for C, T in WINDOWS:
        off.append(sum(a.numel() for a in xs))
        ds_off.append(sum(len(t) for t in tables))
        xs.append(torch.randn(C * T, generator=g, device=cuda))
        # delays of either sign, up to about 40 samples per unit DM
        tables.append(np.linspace(-11.3, 40.7, C).astype(np.float32))
    return torch.cat(xs), torch.from_numpy(np.concatenate(tables)).to(cuda), off, ds_off, tables


def _state(n, cuda, u):
    import torch
    z = dict(dtype=torch.float64, device=cuda)
    return u.clone(), torch.full((n,), 0.1, device=cuda), torch.zeros(n, **z), torch.empty(n, **z), torch.empty(n, **z)


@pytest.mark.parametrize("copies", [1, 60])
@pytest.mark.parametrize("loss_kind", ["energy", "excess"])
def test_evaluation_at_split_edges(cuda, loss_kind, copies):
    """Loss and gradient against the float64 reference; the kernels round the
    interpolation weight to float32 (6e-8), so 1e-5 of the terms' size."""
    import torch
    import frac_ddtr
    x, ds, off, ds_off, tables = _windows(cuda, 3)
    n = len(WINDOWS) * copies
    plan = frac_ddtr.RefinePlan([w[0] for w in WINDOWS] * copies, [w[1] for w in WINDOWS] * copies, off * copies,
                                ds_off * copies, loss=loss_kind)
    for u_val in (0.0, 0.37, -0.81):
        print(f"refine split edges {loss_kind} u={u_val}", flush=True)
        u0 = torch.full((n,), u_val, device=cuda)
        u, step, prev, loss, grad = _state(n, cuda, u0)
        plan.run(x, ds, u, step, prev, loss, grad, nsteps=0)
        torch.cuda.synchronize()
        for v in (loss, grad):   # the copies agree
            assert torch.equal(v.view(copies, -1), v[:len(WINDOWS)].expand(copies, -1))
        for b, (C, T) in enumerate(WINDOWS):
            w = x[off[b]:off[b] + C * T].view(1, C, T).double()
            ub = u0[b:b + 1].double().requires_grad_(True)
            E = (ref.frac_ddtr_torch(w, ub, [0.0], tables[b]) ** 2).sum()
            (gE,) = torch.autograd.grad(E, ub, retain_graph=True)
            N, gN = E.detach() * 0.0, gE * 0.0
            if loss_kind == "excess":
                N = ref.noise_energy_torch(w, ub, tables[b])[0]
                (gN,) = torch.autograd.grad(N, ub)
            scale = float((E + N).detach()) + 1e-12
            gscale = max(abs(float(gE)), abs(float(gN)), 1e-3 * scale)
            assert abs(float(loss[b]) - float((E - N).detach())) <= 1e-5 * scale, (C, T, u_val)
            assert abs(float(grad[b]) - float(gE - gN)) <= 1e-5 * gscale, (C, T, u_val)


@pytest.mark.parametrize("points", [1, 3, 4, 7])
def test_scan_takes_the_best_point(cuda, points):
    import torch
    import frac_ddtr
    x, ds, off, ds_off, _ = _windows(cuda, 4)
    n = len(WINDOWS)
    plan = frac_ddtr.RefinePlan([w[0] for w in WINDOWS], [w[1] for w in WINDOWS], off, ds_off, loss="energy")
    lo, dstep = -0.6, 0.23
    u0 = torch.full((n,), 0.05, device=cuda)
    best_u, best_l = u0, torch.full((n,), -np.inf, dtype=torch.float64, device=cuda)
    for k in range(points):   # every point evaluated by itself; the first of equal ones is kept
        uk = (u0 + np.float32(lo)) + np.float32(np.float32(dstep) * np.float32(k))
        st = _state(n, cuda, uk)
        plan.run(x, ds, *st, nsteps=0)
        better = st[3] > best_l
        best_u, best_l = torch.where(better, uk, best_u), torch.where(better, st[3], best_l)
    st = _state(n, cuda, u0)
    plan.run(x, ds, *st, nsteps=0, scan=(points, lo, dstep))
    torch.cuda.synchronize()
    assert torch.equal(st[0], best_u)
    assert torch.equal(st[3], best_l)
