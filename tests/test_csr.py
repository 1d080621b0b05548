"""The CSR of a plain segment index (fmd_csr_from_index) against a stable sort: exact integers."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def stable_csr(index, num_segment):
    """perm of the rows of [0, num_segment) in stable order and the offsets (NumPy)."""
    order = np.argsort(index, kind="stable")
    inside = order[(index[order] >= 0) & (index[order] < num_segment)]
    count = np.bincount(index[inside], minlength=num_segment)[:num_segment]
    return inside, np.concatenate([[0], np.cumsum(count)])


# one workgroup up to 8192 rows; chunks of 1024 rows above, at most 256 of them (the largest case);
# one pass of 8 bits up to 255 segments, then two and three
@pytest.mark.parametrize("rows,num_segment", [(0, 5), (1, 1), (64, 255), (1023, 256), (2049, 3), (8192, 65536),
                                              (8193, 1), (8193, 255), (30011, 256), (65537, 65536), (300007, 70001),
                                              (0, 20000), (1, 8192), (1, 8193), (1000, 300007)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("kind", ["random", "sorted", "few"])
def test_csr_is_the_stable_order(rows, num_segment, dtype, kind):
    from fastmd_amd.ops.csr_segment_sum import csr_from_segment

    rng = np.random.default_rng(rows + num_segment)
    high = max(1, num_segment // 50) if kind == "few" else num_segment + max(1, num_segment // 100)  # some past the end
    index = rng.integers(0, high, rows)
    if kind == "sorted":
        index = np.sort(index)
    perm, off = stable_csr(index, num_segment)
    strided = torch.tensor(np.stack([index, index + 1], 1), dtype=dtype, device="cuda")[:, 0]
    csr = csr_from_segment(strided, num_segment)
    assert csr.off.cpu().numpy().tolist() == off.tolist()
    assert csr.perm.cpu().numpy()[:off[-1]].tolist() == perm.tolist()
    assert sorted(csr.perm.cpu().numpy().tolist()) == list(range(rows))


def test_more_chunks_from_2_24_rows():
    from fastmd_amd.ops.csr_segment_sum import csr_from_segment

    rows, num_segment = 2 ** 24 + 7, 1_000_003
    index = np.random.default_rng(0).integers(0, num_segment + 10, rows).astype(np.int32)
    perm, off = stable_csr(index, num_segment)
    csr = csr_from_segment(torch.tensor(index, device="cuda"), num_segment)
    assert np.array_equal(csr.off.cpu().numpy(), off) and np.array_equal(csr.perm.cpu().numpy()[:off[-1]], perm)


@pytest.mark.parametrize("rows", [(40, 9000), (9000, 40), (12000, 9000), (40, 8000)])
def test_two_indices_share_the_launches(rows):
    from fastmd_amd.ops.csr_segment_sum import csr_from_segments, refuse_negative

    rng = np.random.default_rng(1)
    sizes = (300, 70000)
    index = [rng.integers(0, n, r) for r, n in zip(rows, sizes)]
    pairs = [(torch.tensor(i, dtype=torch.int32, device="cuda"), n) for i, n in zip(index, sizes)]
    csrs, check = csr_from_segments(pairs)
    refuse_negative(check)
    for csr, i, n in zip(csrs, index, sizes):
        perm, off = stable_csr(i, n)
        assert csr.off.cpu().numpy().tolist() == off.tolist() and csr.perm.cpu().numpy().tolist() == perm.tolist()


@pytest.mark.parametrize("rows", [100, 20000])
def test_negative_segments_are_refused(rows):
    from fastmd_amd.ops.csr_segment_sum import csr_from_segment, csr_segment_sum
    from fastmd_amd.ops.segment import weighted_segment_sum

    index = torch.randint(0, 50, (rows,), device="cuda")
    index[rows // 2] = -1
    value = torch.ones(rows, 4, device="cuda")
    with pytest.raises(RuntimeError):
        csr_from_segment(index, 50)
    with pytest.raises(RuntimeError):
        csr_segment_sum(value, index, 50)
    with pytest.raises(RuntimeError):
        weighted_segment_sum(value, value, index, 50)


@pytest.mark.gpu
def test_negative_flags_are_cleared_between_calls_and_threads():
    """The pooled flags of a refused index do not reach a later check, also with checks of several threads
    and streams open at a time: each reports its own index."""
    from concurrent.futures import ThreadPoolExecutor

    from fastmd_amd.ops.csr_segment_sum import _NegativeCheck, csr_from_segments, refuse_negative

    def one(k):
        bad = k % 3 == 0
        with torch.cuda.stream(torch.cuda.Stream()):
            seg = torch.full((500 + k,), 4, dtype=torch.int32, device="cuda")
            seg[k % 500] = -1 if bad else 2
            for _ in range(3):
                open_checks = [csr_from_segments([(seg, 9)])[1] for _ in range(3)]
                for check in open_checks:
                    if bad:
                        with pytest.raises(RuntimeError, match="non-negative"):
                            refuse_negative(check)
                    else:
                        refuse_negative(check)
        return bad

    one(0)
    one(1)
    with ThreadPoolExecutor(8) as pool:
        assert list(pool.map(one, range(24))) == [k % 3 == 0 for k in range(24)]
    assert all(len(idle) <= _NegativeCheck._KEPT and not any(any(f.tolist()) for f, _ in idle)
               for idle in _NegativeCheck._idle.values())
