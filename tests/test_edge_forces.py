"""fmd_edge_forces_f32 / fmd_tb_edge_forces_f32: the forces formed straight from the rows' geometry gradients,
against the row kernels' gradients summed in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("three_body", [False, True])
@pytest.mark.parametrize("nb,longest,ld", [(8, 20, 8), (8, 40, 12), (8, 20, 9), (5, 33, 5), (16, 100, 16)])
def test_edge_forces(three_body, nb, longest, ld):
    """Runs of no row, of one pass (32 rows) and of several, a run cut by the row count, missing reverse rows, aligned
    and unaligned basis rows. The row gradients are the bits of the row kernel (stored on the real rows only); a
    force is within its number of terms rounding errors of float32 times the sum of magnitudes."""
    from fastmd_amd import _abi

    gen = torch.Generator().manual_seed(nb + longest + ld)
    n, dev = 61, "cuda"
    off = torch.cat([torch.zeros(1, dtype=torch.int64), torch.randint(0, longest + 1, (n,), generator=gen).cumsum(0)])
    real = int(off[-1]) - 1  # the last run is cut
    e_cap = int(off[-1]) + 5
    reverse = torch.randint(-1, real, (e_cap,), generator=gen, dtype=torch.int32)
    rand = lambda *s: torch.randn(*s, generator=gen).to(dev)  # noqa: E731
    geo, de, g0, g1, gg = rand(e_cap, 8), rand(e_cap, nb), rand(e_cap, ld), rand(e_cap, nb), rand(e_cap, 4)
    geo[:, 3] = geo[:, 3].abs() + 1.0
    gu, gfc, gs = rand(e_cap, 3), rand(e_cap), rand(e_cap)
    flags = torch.randint(0, 2, (e_cap,), generator=gen, dtype=torch.uint8).to(dev)
    rows, offd, rev = torch.tensor([real], device=dev), off.to(dev), reverse.to(dev)
    want = torch.empty(e_cap, 3, device=dev)
    forces, gvec = torch.full((n + 1, 3), 7.0, device=dev), torch.full((e_cap, 3), 5.0, device=dev)
    plain = torch.empty(n, 3, device=dev)
    if three_body:
        row = (geo.data_ptr(), de.data_ptr(), nb, g0.data_ptr(), ld, gu.data_ptr(), 3, gfc.data_ptr(), gs.data_ptr(),
               flags.data_ptr())
        names = "fmd_tb_geometry_bwd_f32", "fmd_tb_edge_forces_f32"
    else:
        row = geo.data_ptr(), de.data_ptr(), nb, g0.data_ptr(), ld, g1.data_ptr(), nb, gg.data_ptr()
        names = "fmd_edge_geometry_bwd_f32", "fmd_edge_forces_f32"
    s = _abi.stream_handle()
    _abi.call(names[0], *row, rows.data_ptr(), e_cap, want.data_ptr(), s)
    for out, kept in ((forces, gvec.data_ptr()), (plain, None)):
        _abi.call(names[1], *row, offd.data_ptr(), rev.data_ptr(), rows.data_ptr(), e_cap, n, -1.0, out.data_ptr(), kept,
                  s)
    torch.cuda.synchronize()
    assert torch.equal(gvec[:real], want[:real]) and bool((gvec[real:] == 5.0).all())
    assert torch.equal(plain, forces[:n]) and bool((forces[n] == 7.0).all())
    v, got = want.cpu().double(), forces.cpu().double()
    for i in range(n):
        run = torch.arange(int(off[i]), min(int(off[i + 1]), real))
        back = reverse[run]
        terms = torch.cat([v[back[back >= 0].long()], -v[run]])
        bound = 2.0 ** -23 * max(len(terms), 1) * terms.abs().sum(0)
        assert bool(((got[i] + terms.sum(0)).abs() <= bound).all())
