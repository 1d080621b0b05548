"""fmd_host_report and fmd_count_demand: what the host reads after a build or an evaluation, written by one
kernel into pinned memory."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", [0, 1, 257, 400_003])
def test_host_report(values):
    """Scalars of each width, an energy and a run of floats (past one pass of the largest grid): the same bits;
    what lies behind the outputs is left."""
    from fastmd_amd import _abi

    src = [torch.tensor([201], dtype=torch.uint8), torch.tensor([True]), torch.tensor([-7], dtype=torch.int32),
           torch.tensor([-2 ** 40 - 3], dtype=torch.int64)]
    dev = [t.cuda() for t in src]
    energy = torch.tensor([-1.25e-3], dtype=torch.float64, device="cuda")
    data = torch.randn(max(values, 1), device="cuda")
    out = torch.full((6,), 99, dtype=torch.int64, pin_memory=True)
    out_e = torch.zeros(1, dtype=torch.float64, pin_memory=True)
    out_v = torch.full((values + 3,), 5.0, pin_memory=True)
    _abi.call("fmd_host_report", 4, _abi.ptr_array([t.data_ptr() for t in dev]),
              _abi.array(_abi._i32, [t.element_size() for t in dev]), out.data_ptr(), energy.data_ptr(),
              out_e.data_ptr(), data.data_ptr(), values, out_v.data_ptr(), _abi.stream_handle())
    torch.cuda.synchronize()
    assert out.tolist() == [201, 1, -7, -2 ** 40 - 3, 99, 99]
    assert torch.equal(out_e, energy.cpu()) and torch.equal(out_v[:values], data[:values].cpu())
    assert out_v[values:].tolist() == [5.0] * 3


@pytest.mark.parametrize("n", [1, 63, 1024, 4097, 100_001])
def test_count_demand(n):
    """The largest count and the sum of the clamped ones, exactly, also past 32 bits."""
    from fastmd_amd import _abi

    counts = np.random.default_rng(n).integers(0, 2 ** 20, n).astype(np.int32)
    limit = 2 ** 19
    out = torch.zeros(2, dtype=torch.int64, pin_memory=True)
    dev = torch.tensor(counts, device="cuda")
    _abi.call("fmd_count_demand", dev.data_ptr(), n, limit, out.data_ptr(), _abi.stream_handle())
    torch.cuda.synchronize()
    assert out.tolist() == [int(counts.max()), int(np.minimum(counts, limit).astype(np.int64).sum())]
