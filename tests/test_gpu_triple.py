"""Products on the bf16 matrix cores (gemm_triple.h): three-term operands, all
layouts the same bits, and the fp32 pass for what the terms cannot hold. Every
test asserts which kernel its products took."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import SEED, gemm_tolerance, normwise_rel_err
from vkml_amd import _lib, ops
from vkml_amd import tensor as T
from vkml_amd.device import DeviceArray, DecisionRecorder

pytestmark = pytest.mark.gpu


def _view(x: np.ndarray, how: str) -> DeviceArray:
    """x as a device view: "n" as it lies, "t" stored transposed, "o" inside a
    wider array at an odd offset (rows at any float address), "r" its columns
    stored last to first."""
    swap = list(range(x.ndim - 2)) + [x.ndim - 1, x.ndim - 2]
    if how == "t":
        return DeviceArray.from_numpy(np.ascontiguousarray(x.transpose(swap))).transpose(-2, -1)
    if how == "r":
        d = DeviceArray.from_numpy(np.ascontiguousarray(x[..., ::-1]))
        return DeviceArray(d.shape, d.dtype, d.strides[:-1] + (-1,), d.buffer, x.shape[-1] - 1)
    if how == "o":
        wide = np.full(x.shape[:-1] + (x.shape[-1] + 3,), np.nan, np.float32)
        wide[..., 1:-2] = x
        d = DeviceArray.from_numpy(wide)
        return DeviceArray(x.shape, d.dtype, d.strides, d.buffer, 1)
    return DeviceArray.from_numpy(x)


def _operand_kinds(rec: DecisionRecorder) -> list[str]:
    return [d["chose"] for d in rec.decisions if d["site"] == "matmul.operands"]


def _three_terms(a: DeviceArray, b: DeviceArray, kernel: str | None = None) -> np.ndarray:
    """a @ b, which must run as three-term products (on the given kernel)."""
    with DecisionRecorder() as rec:
        out = ops.matmul(a, b).numpy()
    assert _operand_kinds(rec) == ["three_bf16_terms"]
    took = [d["chose"] for d in rec.decisions if d["site"] == "matmul.kernel"]
    assert took == [kernel] if kernel else took[0].startswith("gemm_triple_")
    return out


def _off(got: np.ndarray, exact: np.ndarray) -> float:
    """The relative error in the 2-norm."""
    return float(np.linalg.norm(got - exact) / np.linalg.norm(exact))


def _bound(k: int) -> float:
    """_off of N(0,1) products: each 16 k round the sum once,
    by at most 2^-24 of a partial sum, whose mean square is half of the last one's
    or less; the roundings are independent. Plus half an ulp of the result. (For
    every k here below 8e-7; a product without its third terms is off by 2.4e-6.)"""
    return 2.0 ** -24 * (1 + 0.5 * np.sqrt(k / 16))


# (kernel, batch, m, n, k): one or three rows or columns past a tile, fewer than
# four rows in the last tile, a last stage of 1, 9 and 15 k, and none
SHAPES = [("64x64", 1, 1000, 1501, 777), ("64x64", 3, 515, 641, 319), ("64x64", 1, 1025, 1089, 1040),
          ("128x128", 1, 4099, 3841, 89), ("128x128", 16, 257, 389, 417), ("128x128", 1, 2051, 3842, 100),
          ("256x128", 16, 257, 897, 257), ("256x128", 16, 1535, 130, 321), ("256x128", 16, 1795, 130, 223)]


@pytest.mark.parametrize("tile,batch,m,n,k", SHAPES)
def test_layouts_and_edges(hip, tile, batch, m, n, k):
    rng = np.random.default_rng(SEED + m + n + k)
    lead = (batch,) if batch > 1 else ()
    a = rng.standard_normal(lead + (m, k), dtype=np.float32)
    b = rng.standard_normal(lead + (k, n), dtype=np.float32)
    print(f"triple {batch} {m}x{n}x{k}", flush=True)
    got = _three_terms(_view(a, "n"), _view(b, "n"), f"gemm_triple_{tile}")
    rows = np.unique(np.r_[0:4, m // 2, m - 4:m])
    exact = a[..., rows, :].astype(np.float64) @ b.astype(np.float64)
    assert _off(got[..., rows, :], exact) <= _bound(k)
    for la, lb in (("n", "t"), ("t", "n"), ("t", "t"), ("o", "o"), ("r", "n"), ("n", "r")):
        same = _three_terms(_view(a, la), _view(b, lb), f"gemm_triple_{tile}")
        differ = int(np.count_nonzero(same.view(np.uint32) != got.view(np.uint32)))
        assert differ == 0, (la, lb)


# the same of sizes that the plan leaves to the fp32 kernels: K split, few tiles
@pytest.mark.parametrize("batch,m,n,k", [(1, 257, 2049, 1025), (1, 67, 130, 40001), (1, 33, 4100, 2100),
                                         (16, 129, 131, 1040)])
def test_layouts_and_edges_of_fp32_products(hip, batch, m, n, k):
    rng = np.random.default_rng(SEED + m + n + k)
    lead = (batch,) if batch > 1 else ()
    a = rng.standard_normal(lead + (m, k), dtype=np.float32)
    b = rng.standard_normal(lead + (k, n), dtype=np.float32)
    print(f"fp32 {batch} {m}x{n}x{k}", flush=True)
    with DecisionRecorder() as rec:
        got = ops.matmul(_view(a, "n"), _view(b, "n")).numpy()
    assert _operand_kinds(rec) == []
    rows = np.unique(np.r_[0:4, m // 2, m - 4:m])
    exact = a[..., rows, :].astype(np.float64) @ b.astype(np.float64)
    assert normwise_rel_err(got[..., rows, :], exact) <= min(gemm_tolerance(k), 2.0 ** -23 * np.sqrt(k))
    for la, lb in (("n", "t"), ("t", "n"), ("t", "t"), ("o", "o"), ("r", "n"), ("n", "r")):
        same = ops.matmul(_view(a, la), _view(b, lb)).numpy()
        assert np.array_equal(same.view(np.uint32), got.view(np.uint32)), (la, lb)


@pytest.mark.parametrize("m,n,k", [(1000, 1501, 777), (4099, 3841, 89), (1000, 700, 600), (2100, 2300, 100)])
@pytest.mark.parametrize("scale_a,scale_b", [(1.0, 1.0), (1e-36, 1e36), (1e30, 1e-30), (3e-39, 1.0), (1e-20, 1e-19)])
def test_scales_keep_fp32_accuracy(hip, m, n, k, scale_a, scale_b):
    """Operands of any fp32 scale, subnormals included: the accuracy of the
    terms, or where they cannot hold the operands of the fp32 pass, whose sum is
    rounded every two k (and one part in 2^24 of the smallest normal number)."""
    rng = np.random.default_rng(SEED + m)
    a = (rng.standard_normal((m, k)) * scale_a).astype(np.float32)
    b = (rng.standard_normal((k, n)) * scale_b).astype(np.float32)
    print(f"triple scale {scale_a} {scale_b}", flush=True)
    ragged = m % 4 != 0 or n % 4 != 0  # the others are left to the fp32 kernels
    got = (_three_terms(_view(a, "n"), _view(b, "n")) if ragged else ops.matmul(_view(a, "n"), _view(b, "n")).numpy())
    got = got[::8].astype(np.float64)
    exact = a[::8].astype(np.float64) @ b.astype(np.float64)
    terms = ragged and min(scale_a, scale_b) > 1e-22  # no input below 2^-110
    assert np.linalg.norm(got - exact) <= (_bound(k if terms else 8 * k) * np.linalg.norm(exact)
                                           + 2.0 ** -149 * k * np.sqrt(exact.size))


def test_lower_terms_below_the_smallest_normal_number(hip):
    """Inputs of 2^-108: their third terms are subnormal bf16 values, which the
    conversion and the matrix cores have to keep (3e-6 of the result if not)."""
    rng = np.random.default_rng(SEED + 1)
    m, n, k = 1000, 1501, 777

    def signed(shape, scale):
        return (rng.uniform(1, 2, shape) * rng.choice([-1, 1], shape) * scale).astype(np.float32)

    a, b = signed((m, k), 2.0 ** -109), signed((k, n), 2.0 ** 100)
    for x, y in ((a, b), (np.ascontiguousarray(b.T), np.ascontiguousarray(a.T))):
        got = _three_terms(_view(x, "n"), _view(y, "n"))[::8]
        exact = x[::8].astype(np.float64) @ y.astype(np.float64)
        assert _off(got, exact) <= _bound(k)


@pytest.mark.parametrize("m,n,k,terms", [(1100, 1300, 801, True), (600, 640, 800, False)])
def test_infinities_nans_and_the_largest_values(hip, m, n, k, terms):
    """Where a 64-bit product is finite in fp32, the result is it; elsewhere
    infinities and NaNs land where IEEE arithmetic puts them."""
    rng = np.random.default_rng(SEED)
    a = rng.uniform(0.5, 1.5, (m, k)).astype(np.float32)
    b = rng.uniform(0.5, 1.5, (k, n)).astype(np.float32)
    a[3, 5] = np.inf
    a[70, 9] = -np.inf
    b[11, 200] = np.nan
    a[130, :] = 0.0
    a[130, 7] = np.finfo(np.float32).max  # rounds up to infinity as a bf16
    b[7, 300] = 0.5
    b[20, 64] = np.inf
    a[200, 20] = 0.0                      # 0 * inf
    got = _three_terms(_view(a, "n"), _view(b, "n")) if terms else ops.matmul(_view(a, "n"), _view(b, "n")).numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        exact = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exact))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(exact))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(exact))
    fine = np.isfinite(exact)
    np.testing.assert_allclose(got[fine], exact[fine], rtol=1e-5)


# forward on the 128x128, 64x64 and 256x128 tiles, weight gradient on 64x64,
# 256x128 and 128x128; one of both left to the fp32 kernels
@pytest.mark.parametrize("n,c,hw,cout,window,stride,forward,backward", [
    (64, 33, (32, 32), 257, 3, 1, 2, 2), (33, 33, (30, 31), 130, 5, 2, 2, 2), (64, 40, (14, 14), 258, 3, 1, 2, 2),
    (37, 40, (19, 23), 70, 3, 1, 2, 0), (9, 65, (30, 31), 130, 5, 2, 0, 2)])
def test_convolutions_are_the_lowered_products(hip, n, c, hw, cout, window, stride, forward, backward):
    rng = np.random.default_rng(SEED + c)
    x = rng.uniform(-1, 1, (n, c) + hw).astype(np.float32)
    w = rng.uniform(-0.1, 0.1, (cout, c, window, window)).astype(np.float32)
    dx, dw = DeviceArray.from_numpy(x), DeviceArray.from_numpy(w)
    pad = window // 2
    print(f"triple conv {x.shape} {cout}", flush=True)
    cols = ops.im2col(dx, window, stride, pad)
    _, ck, L = cols.shape
    with DecisionRecorder() as rec:
        got = ops.conv2d(dx, dw, stride, pad)
        want = ops.matmul(dw.reshape(1, 1, cout, ck).broadcast_to((1, n, cout, ck)), cols.reshape(1, n, ck, L))
    assert _operand_kinds(rec) == ["three_bf16_terms"] * forward
    assert np.array_equal(got.numpy().reshape(-1), want.numpy().reshape(-1))
    g = rng.standard_normal(got.shape).astype(np.float32)
    dg = DeviceArray.from_numpy(g)
    with DecisionRecorder() as rec:
        per = ops.conv2d_weight_grad(dx, dg, window, stride, pad)
        want = ops.matmul(dg.reshape(1, n, cout, L), cols.reshape(1, n, ck, L).transpose(-2, -1)).numpy()
    assert _operand_kinds(rec) == ["three_bf16_terms"] * backward
    assert np.array_equal(per.numpy().reshape(-1), want.reshape(-1))
    total = ops.conv2d_weight_grad_sum(dx, dg, window, stride, pad).numpy()
    exact = np.einsum("nol,nkl->ok", g.reshape(n, cout, L).astype(np.float64), cols.numpy().astype(np.float64),
                      optimize=True)
    assert normwise_rel_err(total, exact) <= 2.0 ** -23 * np.sqrt(n * L)


def test_graph_nodes_keep_the_fp32_kernels(hip):
    """Products and convolutions of a graph, forward and backward, have the
    bits of the fp32 kernels: another order of sums moves a near tie of a
    pool or relu, and the gradients behind it by far more than rounding."""
    rng = np.random.default_rng(SEED + 3)
    x = rng.uniform(-1, 1, (96, 64, 16, 16)).astype(np.float32)
    w = rng.uniform(-0.05, 0.05, (128, 64, 3, 3)).astype(np.float32)
    u, v = rng.standard_normal((1000, 777)).astype(np.float32), rng.standard_normal((1501, 777)).astype(np.float32)
    with DecisionRecorder() as rec:
        tx, tw = T.tensor(x, requires_grad=True), T.tensor(w, requires_grad=True)
        y = T.conv2d(tx, tw, padding=1)
        T.backward(T.sum(y))
        tu, tv = T.tensor(u, requires_grad=True), T.tensor(v, requires_grad=True)
        z = T.matmul(tu, tv.transpose(-2, -1))
        T.backward(T.sum(z))
        got = [t.numpy() for t in (y, tx.grad, tw.grad, z, tu.grad, tv.grad)]
    assert _operand_kinds(rec) == []
    # plans of one partition: split_k=1 is the fp32 kernel of the same plan
    assert ops.gemm_plan(96, 128, 256, 576)[0] == ops.gemm_plan(1, 1000, 1501, 777)[0] == 1
    cols = ops.im2col(DeviceArray.from_numpy(x), 3, 1, 1).reshape(1, 96, 576, 256)
    flat = DeviceArray.from_numpy(w.reshape(1, 1, 128, 576)).broadcast_to((1, 96, 128, 576))
    assert np.array_equal(got[0].reshape(-1), ops.matmul(flat, cols, split_k=1).numpy().reshape(-1))
    assert np.array_equal(got[3], ops.matmul(_view(u, "n"), _view(v, "n").T, split_k=1).numpy())
    ones = np.ones((1000, 1501))
    for grad, exact in ((got[4], ones @ v), (got[5], ones.T @ u)):
        assert normwise_rel_err(grad, exact) <= gemm_tolerance(1501)


def test_a_forced_kernel_or_split_stays_on_the_fp32_cores(hip):
    rng = np.random.default_rng(SEED + 5)
    a, b = (_view(rng.standard_normal(s).astype(np.float32), "n") for s in ((1000, 777), (777, 1501)))
    auto = _three_terms(a, b)
    with DecisionRecorder() as rec:
        forced = ops.matmul(a, b, kernel=_lib.GEMM_MFMA).numpy()
        unsplit = ops.matmul(a, b, split_k=1).numpy()
    assert _operand_kinds(rec) == []
    assert ops.gemm_plan(1, 1000, 1501, 777)[0] == 1 and np.array_equal(forced, unsplit)
    assert not np.array_equal(forced, auto)


def test_sums_of_one_term_are_rounded_as_in_fp32(hip):
    """A diagonal matrix times a matrix is one product per output. The operands'
    lower terms are as large as they get (1 + 2^-8 - 2^-17 and its neighbours),
    so every term product but l * l' (2^-34 of the product) shows: half an ulp,
    2^-24, plus that and its few roundings."""
    n = 2048
    d = np.full(n, 0x3f807fc0, np.int32).view(np.float32)
    b = (0x3f807fc0 + np.arange(-n // 2, n // 2, dtype=np.int32)).view(np.float32)
    b = np.broadcast_to(b, (n, n)).copy()
    got = _three_terms(_view(np.diag(d), "n"), _view(b, "n"))
    exact = d.astype(np.float64)[:, None] * b.astype(np.float64)
    assert np.max(np.abs(got - exact) / exact) <= 2.0 ** -24 * (1 + 2.0 ** -7)


# (128x128 and 256x128 tiles, ragged rows, a last stage of 4 and of 1 k; pairs of
# partitions)
@pytest.mark.parametrize("batch,m,n,k,terms", [(1, 336, 422, 20164, True), (1, 448, 691, 20308, True),
                                               (4, 210, 446, 7473, True), (1, 304, 208, 34936, False)])
@pytest.mark.parametrize("one_sign", [False, True])
def test_split_plans_keep_their_partitions(hip, batch, m, n, k, terms, one_sign):
    """A product whose K the plan splits is summed partition by partition, in
    chains no longer than the fp32 kernels': no less exact than those, also
    where every product is of one sign, in every layout the same bits."""
    splits, chunk = ops.gemm_plan(batch, m, n, k)
    assert splits > 2
    rng = np.random.default_rng(SEED + 7)
    lead = (batch,) if batch > 1 else ()
    a, b = (rng.standard_normal(lead + s).astype(np.float32) for s in ((m, k), (k, n)))
    if one_sign:
        a, b = np.maximum(a, 0), np.maximum(b, 0)
    with DecisionRecorder() as rec:
        got = ops.matmul(_view(a, "n"), _view(b, "n")).numpy()
    assert _operand_kinds(rec) == ["three_bf16_terms"] * terms
    assert [d["chose"] for d in rec.decisions if d["site"] == "matmul.split_k"] == [f"split_k_{splits}"]
    rows = np.arange(0, m, 16)
    fp32 = ops.matmul(_view(a, "n"), _view(b, "n"), kernel=_lib.GEMM_MFMA).numpy()[..., rows, :]
    exact = a[..., rows, :].astype(np.float64) @ b.astype(np.float64)
    assert _off(got[..., rows, :], exact) <= _off(fp32, exact)
    for la, lb in (("n", "t"), ("t", "n"), ("o", "o"), ("r", "n")):
        same = ops.matmul(_view(a, la), _view(b, lb)).numpy()
        assert np.array_equal(same.view(np.uint32), got.view(np.uint32)), (la, lb)


@pytest.mark.parametrize("n,c,hw,cout,window", [(70, 33, (24, 20), 250, 3), (40, 40, (24, 24), 200, 5)])
def test_weight_gradients_summed_over_a_batch(hip, n, c, hw, cout, window):
    """The batch folded into K, ragged rows and columns: each partition a chain,
    and a fold that rounds log2(partitions) times."""
    rng = np.random.default_rng(SEED + c)
    x = rng.uniform(-1, 1, (n, c) + hw).astype(np.float32)
    g = rng.standard_normal((n, cout) + hw).astype(np.float32)
    k, ck = n * hw[0] * hw[1], c * window * window
    splits, chunk = ops.gemm_plan(1, cout, ck, k)
    dx, dg = DeviceArray.from_numpy(x), DeviceArray.from_numpy(g)
    with DecisionRecorder() as rec:
        got = ops.conv2d_weight_grad_sum(dx, dg, window, 1, window // 2).numpy()
    assert _operand_kinds(rec) == ["three_bf16_terms"]
    cols = ops.im2col(dx, window, 1, window // 2).numpy()
    exact = np.zeros((cout, ck))
    for image in range(n):
        exact += g[image].reshape(cout, -1).astype(np.float64) @ cols[image].astype(np.float64).T
    assert _off(got, exact) <= _bound(32 * chunk) + 2.0 ** -24 * np.sqrt(np.log2(splits))


def test_tiny_inputs_among_ordinary_ones_change_nothing(hip):
    """Inputs below 2^-110 lose low bits as terms, nothing beside outputs of
    ordinary size: those keep the bits they have with zeros in their place. An
    output made of such inputs alone has fp32's accuracy."""
    rng = np.random.default_rng(SEED + 9)
    m, n, k = 1000, 1501, 777
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a[:, 5] = 0.0
    want = _three_terms(_view(a, "n"), _view(b, "n"))
    a[::7, 5] = 1e-36
    b[3, ::11] *= np.float32(1e-38)
    zeroed = b.copy()
    zeroed[3, ::11] = 0.0
    want[:, ::11] = _three_terms(_view(a, "n"), _view(zeroed, "n"))[:, ::11]
    got = _three_terms(_view(a, "n"), _view(b, "n"))
    assert np.count_nonzero(got.view(np.uint32) != want.view(np.uint32)) == 0
    a[130] = rng.standard_normal(k) * 1e-35
    got = _three_terms(_view(a, "n"), _view(b, "n"))
    exact = a[130].astype(np.float64) @ b.astype(np.float64)
    assert _off(got[130], exact) <= _bound(8 * k)  # the fp32 pass rounds every two k


def test_decisions_name_the_kernel_that_runs(hip):
    a, b = DeviceArray((1000, 777)), DeviceArray((777, 1501))
    with DecisionRecorder() as rec:
        ops.matmul(a, b)
    by_site = {d["site"]: d for d in rec.decisions}
    kernel = by_site["matmul.kernel"]
    assert (kernel["chose"], kernel["instead_of"]) == ("gemm_triple_64x64", "gemm_mfma_64x64")
    assert (kernel["required"], kernel["available"]) == (16 * 24, hip.capabilities().compute_units)
    operands = by_site["matmul.operands"]
    assert (operands["required"], operands["available"], operands["dispatch"]) == (1000, 1501, kernel["dispatch"])
    assert "matmul.split_k" not in by_site
