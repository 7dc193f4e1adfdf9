"""Fractional-delay forward pass and DM adjoint with the channels split over
work-groups (small batches), against the float64 reference: channel counts
around whole chunks (12) and parts, one and several trial groups."""
import numpy as np
import pytest

import frac_ddtr_ref as ref

pytestmark = pytest.mark.gpu


# batch, channels, samples, trials
@pytest.mark.parametrize("shape", [(1, 191, 64, 5), (1, 192, 128, 33), (2, 193, 1028, 16), (1, 1541, 256, 16),
                                   (3, 1548, 64, 64), (1, 4096, 4, 1), (5, 40, 64, 3)])
def test_split_channels_match_reference(cuda, shape):
    """Forward within 2e-6 and DM gradient within 1e-5 of the result's size:
    float32 sums of up to 4096 channels, as for the unsplit kernels."""
    import torch
    import frac_ddtr
    B, C, T, K = shape
    print(f"frac split {shape}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(B * C + T)
    ds = np.linspace(0.0, 3.7, C).astype(np.float32)
    trials = np.linspace(-2.0, 2.0, K).astype(np.float32)
    x = torch.randn((B, C, T), generator=g, device=cuda, requires_grad=True)
    dm = (torch.rand(B, generator=g, device=cuda) - 0.5).requires_grad_(True)
    plan = frac_ddtr.FracPlan(ds, trials, T, B)
    y = frac_ddtr.frac_dedisperse(x, dm, plan)
    gy = torch.randn(y.shape, generator=g, device=cuda)
    gx, gdm = torch.autograd.grad((y * gy).sum(), (x, dm))
    x64, dm64 = x.detach().double().requires_grad_(True), dm.detach().double().requires_grad_(True)
    y64 = ref.frac_ddtr_torch(x64, dm64, trials.astype(np.float64), ds.astype(np.float64))
    gx64, gdm64 = torch.autograd.grad((y64 * gy.double()).sum(), (x64, dm64))
    scale = float(y64.detach().abs().max())
    assert float((y.double() - y64).abs().max()) <= 2e-6 * scale * max(1.0, (C / 256) ** 0.5)
    assert float((gx.double() - gx64).abs().max()) <= 2e-6 * float(gx64.abs().max())
    assert float((gdm.double() - gdm64).abs().max()) <= 1e-5 * max(float(gdm64.abs().max()), scale)


def test_two_streams_share_a_plan(cuda):
    """Forward and backward of one plan on two streams at once give, bit for bit,
    what they give alone."""
    import torch
    import frac_ddtr
    B, C, T, K = 2, 2048, 1024, 32
    g = torch.Generator(device=cuda).manual_seed(3)
    plan = frac_ddtr.FracPlan(np.linspace(0.0, 3.7, C).astype(np.float32), np.linspace(-2.0, 2.0, K), T, B)
    xs = [torch.randn((B, C, T), generator=g, device=cuda, requires_grad=True) for _ in range(2)]
    dms = [(torch.rand(B, generator=g, device=cuda) - 0.5).requires_grad_(True) for _ in range(2)]

    def step(i):
        y = frac_ddtr.frac_dedisperse(xs[i], dms[i], plan)
        return [y.detach()] + list(torch.autograd.grad(y.square().sum(), (xs[i], dms[i])))

    want = [step(i) for i in range(2)]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in range(2)], [[], []]
    for _ in range(10):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(step(i))
    torch.cuda.synchronize()
    for i in range(2):
        for result in got[i]:
            for a, b in zip(result, want[i]):
                assert torch.equal(a, b)
