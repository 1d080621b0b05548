"""float32 gemm whose B is split into bf16 planes by the call itself (b [K, N], and large b [N, K]):
every width of the last column tile against float64, and non-finite operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(a, b, b_layout):
    return a.double() @ (b.double().t() if b_layout == 0 else b.double())


# last column tiles of 8, 32, 33, 64, 65 and 128 columns; K of one partial slice, of an odd number of 16-k slices
# and of exact ones; the smallest row counts of the route
@pytest.mark.parametrize("m,n,k", [(32641, 40, 20), (16257, 136, 264), (10900, 288, 36), (10900, 289, 48),
                                   (8129, 448, 64), (8129, 449, 100), (6600, 520, 1024), (32700, 128, 260)])
@pytest.mark.parametrize("form", ["plain", "bias_silu", "accumulate"])
def test_b_layout_1(m, n, k, form):
    from fastmd_amd.ops import wide_gemm

    assert wide_gemm._takes_planes(m, n, k, 1)
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k + 4, generator=gen, device="cuda")[:, :k]  # a row stride of its own
    b = torch.randn(k, n + 3, generator=gen, device="cuda")[:, :n]
    want = reference(a, b, 1)
    if form == "bias_silu":
        bias = torch.randn(n, generator=gen, device="cuda")
        got = wide_gemm.gemm(a, b, b_layout=1, bias=bias, epilogue="silu")
        want = torch.nn.functional.silu(want + bias.double())
    elif form == "accumulate":
        out = torch.randn(m, n, generator=gen, device="cuda")
        want = want + out.double()
        got = wide_gemm.gemm(a, b, b_layout=1, out=out, accumulate=True)
    else:
        got = wide_gemm.gemm(a, b, b_layout=1)
    # three planes per operand: 2^-24 per product, K products summed in fp32; 1e-5 of the largest element as
    # for every float32 gemm here
    assert float((got.double() - want).abs().max()) <= 1e-5 * float(want.abs().max())


# either side of every line of the choice, by rows, tiles, K and the last column tile
@pytest.mark.parametrize("m,n,k,b_layout,planes", [
    (65600, 40, 20, 1, True), (65400, 40, 20, 1, False), (32700, 40, 188, 1, False), (32700, 40, 192, 1, True),
    (16300, 136, 44, 1, False), (16300, 136, 48, 1, True), (16300, 256, 20, 1, True), (26000, 168, 20, 1, True),
    (24300, 168, 64, 1, False), (24700, 160, 20, 1, True), (24000, 160, 20, 1, False), (49200, 24, 20, 1, False),
    (255, 65536, 20, 1, False), (256, 49152, 20, 1, True), (383, 16384, 64, 1, False), (385, 16384, 64, 1, True),
    (16384, 1024, 1028, 0, True), (16383, 1024, 1028, 0, False)])
def test_choice_of_the_form(monkeypatch, m, n, k, b_layout, planes):
    from fastmd_amd import _abi
    from fastmd_amd.ops import wide_gemm

    taken, call = [], _abi.call
    monkeypatch.setattr(_abi, "call", lambda name, *args: (taken.append(name), call(name, *args))[1])
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, generator=gen, device="cuda")
    b = torch.randn(*((k, n) if b_layout else (n, k)), generator=gen, device="cuda")
    got, want = wide_gemm.gemm(a, b, b_layout=b_layout), reference(a, b, b_layout)
    assert taken == ["fmd_gemm_f32_planes" if planes else "fmd_gemm_f32"]
    assert float((got.double() - want).abs().max()) <= 1e-5 * float(want.abs().max())


def test_large_b_layout_0_equals_the_kernel_that_splits_both():
    """The same planes and K order: bitwise gemm_gather, which splits B in the kernel."""
    from fastmd_amd.ops import wide_gemm

    m, n, k = 160000, 392, 280  # a last column tile of 8
    assert wide_gemm._takes_planes(m, n, k, 0)
    gen = torch.Generator(device="cuda").manual_seed(1)
    a, b = torch.randn(m, k, generator=gen, device="cuda"), torch.randn(n, k, generator=gen, device="cuda")
    assert torch.equal(wide_gemm.gemm(a, b, b_layout=0), wide_gemm.gemm_gather([(a, None)], b))


# b [K, N] and, from 2^34 multiply-adds, b [N, K] through the planes; both in the fp32 form below 256 tiles
@pytest.mark.parametrize("n,m,k,b_layout", [(128, 32700, 64, 1), (136, 32700, 64, 1), (520, 33000, 1024, 0),
                                            (136, 2000, 64, 0), (136, 2000, 64, 1)])
def test_non_finite_operands_follow_the_fp32_product(n, m, k, b_layout):
    """Infinities, NaN and values that round to an infinite bf16 give what float64 gives (an infinity
    kept, inf - inf and inf * 0 NaN), and leave the other rows and columns alone."""
    from fastmd_amd.ops import wide_gemm

    gen = torch.Generator(device="cuda").manual_seed(2)
    a, b = torch.randn(m, k, generator=gen, device="cuda"), torch.randn(k, n, generator=gen, device="cuda")
    b[:, 3] = b[:, 3].to(torch.bfloat16).float()  # its lower planes are zero
    a[:, 5] *= 1e-3  # the products of the large finite values stay finite
    b[2] *= 1e-3
    a[5, 7], a[6, 7], a[6, 9], a[7, 1], a[8, 2] = float("inf"), float("inf"), float("-inf"), float("nan"), 3.4e38
    b[4, n - 1], b[5, n - 2] = float("inf"), 3.4e38
    a[9, 4] = 0.0  # times that infinity
    b = b if b_layout else b.t().contiguous()
    assert wide_gemm._takes_planes(m, n, k, b_layout) == (m > 2000)
    want = reference(a, b, b_layout)
    got = wide_gemm.gemm(a, b, b_layout=b_layout).double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    fine = torch.isfinite(want) & (want.abs() < 1e30)
    assert float((got - want)[fine].abs().max()) <= 1e-5 * float(want[fine].abs().max())
    big = torch.isfinite(want) & ~fine
    assert float(((got - want)[big] / want[big]).abs().max()) <= 1e-5


def test_non_finite_gathered_parts():
    """Rows gathered from two sources and K in three parts: an infinity in each, the rows that gather them and no other."""
    from fastmd_amd.ops import wide_gemm

    m, n = 33000, 136
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, y, z = (torch.randn(r, w, generator=gen, device="cuda") for r, w in ((700, 48), (900, 16), (m, 20)))
    w = torch.randn(n, 84, generator=gen, device="cuda")
    x[5, 7], y[11, 3], z[17, 19] = float("inf"), float("-inf"), float("nan")
    i, j = (torch.randint(0, r, (m,), generator=gen, device="cuda", dtype=torch.int32) for r in (700, 900))
    want = reference(torch.cat([x[i.long()], y[j.long()], z], 1), w, 0)
    parts = [(x, i), (y, j), (z, None)]
    got = wide_gemm.gemm_planes(parts, wide_gemm.split_planes(w), a_planes=False).double()
    fine = torch.isfinite(want)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()]) and bool(got.isinf().any())
    # split in the kernel: not finite in the same places, the same values elsewhere
    inside = wide_gemm.gemm_gather(parts, w).double()
    assert torch.equal(torch.isfinite(inside), fine)
    for x in (got, inside):
        assert float((x - want)[fine].abs().max()) <= 1e-5 * float(want[fine].abs().max())


# the third plane of an operand of 2^e has a step of 2^-133 (bf16's smallest): 24 bits down to e = -110, 24 - 8 from
# there to -118; the fp32 form keeps 24 down to fp32's own range
@pytest.mark.parametrize("exponent,bits", [(-100, 24), (-110, 24), (-118, 16)])
def test_small_operands(exponent, bits):
    from fastmd_amd.ops import wide_gemm

    m, n, k = 33000, 256, 64
    assert wide_gemm._takes_planes(m, n, k, 1) and wide_gemm._planes_pay(m, n, k, 1)
    gen = torch.Generator(device="cuda").manual_seed(-exponent)
    a = (1.0 + torch.rand(m, k, generator=gen, device="cuda")) * 2.0 ** exponent
    b = 1.0 + torch.rand(k, n, generator=gen, device="cuda")
    want = reference(a, b, 1)
    worst = float(((wide_gemm.gemm(a, b, b_layout=1).double() - want) / want).abs().max())
    print(f"[small operands] 2^{exponent}: {worst:.2e}", flush=True)
    # positive terms: the operand's own error plus K roundings of the sum
    assert worst <= 2.0 ** -(bits - 1) + k * 2.0 ** -24


def test_infinities_in_every_row():
    """A blown-up input: every output element that is not finite is what float64 says, and the product is formed within
    20 times the time of a finite one (blocks of it are formed twice; element by element it took several hundred)."""
    from fastmd_amd.ops import wide_gemm

    m, n, k = 65600, 128, 512
    gen = torch.Generator(device="cuda").manual_seed(3)
    a, b = torch.randn(m, k, generator=gen, device="cuda"), torch.randn(k, n, generator=gen, device="cuda")
    bad = a.clone()
    bad[torch.arange(m), torch.arange(m) % k] = float("inf")
    bad[::5, 3] = float("-inf")
    want, got = reference(bad, b, 1), wide_gemm.gemm(bad, b, b_layout=1).double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()]) and bool(want.isnan().any()) and bool(want.isinf().any())

    def best(x):
        out, times = torch.empty(m, n, device="cuda"), []
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            wide_gemm.gemm(x, b, b_layout=1, out=out)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    finite, blown = best(a), best(bad)
    print(f"[infinities] finite {finite * 1e3:.0f} us, blown up {blown * 1e3:.0f} us", flush=True)
    assert blown <= 20 * finite
