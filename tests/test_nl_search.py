"""The candidate search's forms (a wave per atom, a workgroup per atom, both in one refresh), rows
refreshed over old rows, and the Morton order on the GPU against the host's."""
import numpy as np
import pytest
import torch

from fastmd_amd.adapters.protocol import PaddingRule
from oracle import nl as onl

pytestmark = pytest.mark.gpu
F32 = np.float32


def builder_of(cell, n, device, cutoff=6.0, skin=2.0):
    from fastmd_amd.graph.fixed_capacity_builder import FixedCapacityGraphBuilder

    return FixedCapacityGraphBuilder(cell=torch.tensor(cell, dtype=torch.float32), atomic_numbers=torch.ones(n),
                                     u_capacity=64, t_capacity=0, line_graph_cutoff=None, atom_graph_cutoff=cutoff,
                                     candidate_cutoff=cutoff + skin, padding=PaddingRule("far_self_loops"), device=device)


def assert_rows(builder, positions, cell):
    cell32 = cell.astype(F32)
    _, _, wrapped = onl.wrap(positions, builder.inv_cell.cpu().numpy(), cell32)
    cand = onl.candidates(wrapped, cell32, F32(builder._cand2), builder.buffer_max)
    assert np.array_equal(builder.num_neighbors.cpu().numpy(), cand.num_neighbors)
    assert np.array_equal(builder.neighbor_matrix.cpu().numpy(), cand.neighbor_matrix)
    assert np.array_equal(builder.neighbor_shifts.cpu().numpy(), cand.neighbor_shifts)
    assert bool(builder._candidate_capacity_valid.item()) == cand.capacity_valid
    return cand.num_neighbors


def spread(n, cell, seed):
    return np.random.default_rng(seed).uniform(0, 1, (n, 3)) @ cell


def clustered(n, cell, dense, seed):
    """``dense`` of the atoms inside a ball, the rest anywhere."""
    positions = spread(n, cell, seed)
    rng = np.random.default_rng(seed + 1)
    v = rng.normal(size=(dense, 3))
    positions[:dense] = 15.0 + 3.5 * v / np.linalg.norm(v, axis=1, keepdims=True) * rng.uniform(0, 1, (dense, 1)) ** (1 / 3)
    return positions


# per refresh: everything in the wave form; rows of up to 64, above 64 and above 256 candidates (the last by the
# workgroup form behind it); and back, each over the rows of the one before
@pytest.mark.parametrize("shear", [0.0, 0.2])
def test_rows_over_old_rows(device, shear):
    cell = np.diag([41.0, 37.0, 33.0])
    cell[1, 0] = shear * 37.0
    n = 700
    builder = builder_of(cell, n, device)
    sizes = []
    for positions in (spread(n, cell, 0), clustered(n, cell, 120, 1), clustered(n, cell, 300, 2), spread(n, cell, 3),
                      clustered(n, cell, 257, 4)):
        builder.refresh_candidates(torch.tensor(positions, device=device))
        sizes.append(int(assert_rows(builder, positions, cell).max()))
    assert sizes[0] <= 64 < sizes[1] <= 256 < sizes[2] and sizes[3] <= 64


def test_dense_rows_take_the_workgroup_form(device):
    """A mean row near the wave form's keys: every row by the workgroup form, over old rows."""
    cell = np.eye(3) * 17.0
    n = 600
    builder = builder_of(cell, n, device)
    for seed in (0, 1):
        positions = spread(n, cell, seed)
        builder.refresh_candidates(torch.tensor(positions, device=device))
        assert int(assert_rows(builder, positions, cell).min()) > 150


@pytest.mark.parametrize("n,side,cutoff", [(5, 4.5, 11.0), (8, 4.0, 7.0), (40, 9.0, 11.0), (11, 9.0, 11.0)])
def test_cells_thinner_than_the_cutoff(device, n, side, cutoff):
    """One cell per axis searched over two images and more: rows above the wave form's keys from few atoms
    (the first three), and below."""
    cell = np.diag([side, side, side * 1.03])
    builder = builder_of(cell, n, device, cutoff=cutoff, skin=1.0)
    assert max(builder._reach) > 1
    for seed in (0, 1):
        positions = spread(n, cell, seed)
        builder.refresh_candidates(torch.tensor(positions, device=device))
        assert (int(assert_rows(builder, positions, cell).max()) > 256) == (n != 11)


def test_slab_in_vacuum(device):
    """A mean density of the wave form, rows of the workgroup form: left unsearched inside, ended early near the
    surface; then over those rows a spread system and back."""
    cell = np.diag([30.0, 30.0, 120.0])
    n = 1700
    builder = builder_of(cell, n, device, cutoff=8.0)
    slab = np.diag([30.0, 30.0, 20.0])
    for seed, box in ((0, slab), (1, cell), (2, slab)):
        positions = spread(n, box, seed)
        builder.refresh_candidates(torch.tensor(positions, device=device))
        rows = assert_rows(builder, positions, cell)
        assert rows.max() > 256 and rows.min() < 256 if box is slab else rows.max() <= 256


def test_full_cells_with_short_rows_keep_the_capacity_flag(device):
    """27 tight clusters within reach of each other's cells but not of the cutoff: more atoms in the cells than the
    wave form expects to hold, rows that fit the slots."""
    cell = np.eye(3) * 60.0
    side = 60.0 / 7
    centre = side * 3.5 + 12.0 * (np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 3) - 1)
    rng = np.random.default_rng(0)
    positions = (centre[:, None] + rng.uniform(-0.2, 0.2, (27, 100, 3))).reshape(-1, 3)
    n, slots = len(positions), 128
    builder = builder_of(cell, n, device)
    assert tuple(builder._ncells) == (7, 7, 7)
    builder.buffer_max = slots
    builder.neighbor_matrix = torch.full((n, slots), n, dtype=torch.int32, device=device)
    builder.neighbor_shifts = torch.zeros((n, slots, 3), dtype=torch.int32, device=device)
    builder.refresh_candidates(torch.tensor(positions, device=device))
    assert int(assert_rows(builder, positions, cell).max()) == 99
    assert bool(builder._candidate_capacity_valid.item())


@pytest.mark.parametrize("skin,slots", [(0.5, 16), (2.0, 48)])
def test_truncated_rows_of_the_wave_form(device, skin, slots):
    """More candidates than slots: the first in order, the flag cleared."""
    cell = np.diag([41.0, 37.0, 33.0])
    n = 900
    builder = builder_of(cell, n, device, skin=skin)
    builder.buffer_max = slots
    builder.neighbor_matrix = torch.full((n, slots), n, dtype=torch.int32, device=device)
    builder.neighbor_shifts = torch.zeros((n, slots, 3), dtype=torch.int32, device=device)
    for seed in (0, 1):
        positions = clustered(n, cell, 60, seed)
        builder.refresh_candidates(torch.tensor(positions, device=device))
        assert int(assert_rows(builder, positions, cell).max()) > slots


@pytest.mark.parametrize("n", [1, 63, 4000, 8192, 8193, 30001])
def test_morton_order_equals_the_host(n):
    from fastmd_amd.graph.fixed_capacity_builder import morton_order

    frac = torch.rand(n, 3, generator=torch.Generator().manual_seed(n))
    frac[::7] = frac[0].clone()  # equal codes keep their order
    frac[n // 2] = torch.tensor([0.0, 1.0 - 2.0 ** -24, 0.5])
    assert torch.equal(morton_order(frac.cuda()).cpu(), morton_order(frac))


@pytest.mark.parametrize("repeats", [(1, 1, 1), (2, 2, 2), (2, 2, 3), (1, 1, 13)])
@pytest.mark.parametrize("short", [0, 40])
def test_build_on_either_side_of_the_fused_form(device, repeats, short):
    """5, 40, 60 atoms in one workgroup (the most of that form), 65 in three launches: every published
    buffer bit-exact against the oracle, with rows to spare and with too few."""
    from test_nl import _assert_build_equal, _oracle_build

    from fastmd_amd import systems
    from fastmd_amd.graph.fixed_capacity_builder import FixedCapacityGraphBuilder

    s = systems.perovskite(repeats)
    pairs = 9 * s.n_atoms - short // 2 * (s.n_atoms // 10)
    builder = FixedCapacityGraphBuilder(cell=torch.tensor(s.cell, dtype=torch.float32), t_capacity=0,
                                        atomic_numbers=torch.ones(s.n_atoms), u_capacity=pairs,
                                        line_graph_cutoff=None, atom_graph_cutoff=6.0, candidate_cutoff=8.0,
                                        padding=PaddingRule("far_self_loops"), device=device)
    rng = np.random.default_rng(0)
    cand, _, _ = _oracle_build(s.cell, s.positions, 6.0, 2.0, builder.e_capacity, inv=builder.inv_cell.cpu().numpy())
    builder.refresh_candidates(torch.tensor(s.positions, device=device))
    moved = s.positions + rng.normal(0, 0.1, s.positions.shape)
    builder.build(torch.tensor(moved, device=device), rebuild_candidates=False)
    _, ob, _ = _oracle_build(s.cell, moved, 6.0, 2.0, builder.e_capacity, ref_positions=s.positions,
                             inv=builder.inv_cell.cpu().numpy())
    _assert_build_equal(builder, ob, cand)
    assert short == 0 or s.n_atoms < 10 or bool(builder._overflow.item())
