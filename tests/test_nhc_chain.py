"""The single-workgroup NHC kernels at the edges of their register forms (atoms per thread, links held)
and with exponents on both sides of the polynomial's range, against the float64 oracle; the fused
post / pre launch against the separate halves, bitwise."""
import numpy as np
import pytest
import torch

from fastmd_amd import units
from oracle import nhc as onhc

pytestmark = pytest.mark.gpu


# (atoms, links, loops, damping in fs, time step in fs): 1, 2, 4, 8 and 16 atoms per thread of 256; up to 4 links and
# up to 8; a strong thermostat, whose exponents pass 2^-5
@pytest.mark.parametrize("n,tchain,tloop,tdamp,dt", [(1, 3, 1, 25.0, 0.25), (256, 4, 1, 25.0, 0.25),
                                                     (257, 5, 1, 25.0, 0.25), (512, 1, 2, 25.0, 0.25),
                                                     (1024, 8, 1, 25.0, 0.25), (1025, 3, 1, 25.0, 0.25),
                                                     (2049, 3, 2, 25.0, 0.25), (4096, 2, 1, 25.0, 0.25),
                                                     (135, 3, 1, 2.0, 2.0), (300, 6, 3, 1.5, 2.0)])
def test_chain_forms(device, n, tchain, tloop, tdamp, dt):
    from fastmd_amd.execution.gpu_nhc import GPUNoseHooverChainNVT, maxwell_boltzmann_momenta

    rng = np.random.default_rng(n)
    masses, q0 = rng.uniform(20.0, 140.0, n), rng.uniform(0.0, 10.0, (n, 3))
    p = maxwell_boltzmann_momenta(masses, 700.0, seed=1)
    force = onhc.harmonic(q0 + 0.1, 0.3)
    f0, e0 = force(q0)
    kw = dict(temperature_K=500.0, timestep=dt * units.fs, tdamp=tdamp * units.fs, tchain=tchain, tloop=tloop)
    o = onhc.NHC(masses, q0, p, forces=f0, energy=e0, **kw)
    g, fused = (GPUNoseHooverChainNVT(masses, q0, p, forces=f0, potential_energy=e0, device=device, **kw) for _ in range(2))
    centre = torch.tensor(q0 + 0.1, device=device)
    q = fused.step_pre_force()
    largest = 0.0
    for step in range(10):
        o.step(force)
        largest = max(largest, float(np.abs(o.p_eta[1:] / o.Q[1:]).max(initial=0.0)) * max(abs(s[2]) for s in o.sub))
        g.step_post_force(-0.3 * (g.step_pre_force() - centre), energy=torch.zeros(1, dtype=torch.float64, device=device))
        if step < 9:
            q = fused.step_post_pre(-0.3 * (q - centre), energy=torch.zeros(1, dtype=torch.float64, device=device))
    fused.step_post_force(-0.3 * (q - centre), energy=torch.zeros(1, dtype=torch.float64, device=device))
    assert tdamp > 10 or largest > 0.03125  # the general exponential ran too
    a, b = g.state.numpy(), fused.state.numpy()
    for name, ref in (("positions", o.q), ("momenta", o.p), ("eta", o.eta), ("p_eta", o.p_eta)):
        assert np.array_equal(a[name], b[name]), name
        # 1e-12 of the largest, as for the other NHC parity tests (float64 rounding over 10 steps)
        assert np.max(np.abs(a[name] - ref)) <= 1e-12 * np.max(np.abs(ref)), name
