"""Contractions of extents and strides that are not multiples of a vector or a tile, on the matrix cores:
against a float64 recomputation from the same inputs.  Both operands bf16: products are exact and summed in
fp32; an fp32 operand keeps all its bits (a mixed product is computed in fp32)."""
import numpy as np
import pytest

from ocannl_amd import backend
from ocannl_amd import llir as L
from ocannl_amd import workloads as W
from parity import HipRun, OracleRun
from test_contract_any_cpu import _same_numbers, gathered_then_multiplied, input_gradient, non_finite
from test_gpu_contractions import _routine
from test_gpu_conv import _conv

pytestmark = pytest.mark.gpu


def _values(rng, node):
    return W.as_prec(rng.standard_normal(node.dims).astype(np.float32), node.prec)


def _run(r, nodes, out, want, accumulate, k, seed=0):
    """`want`: float64 inputs by name -> result without the accumulated-into values."""
    rng = np.random.default_rng(seed)
    init = {n.id: _values(rng, n) for n in nodes.values()}
    hip = HipRun(r, init, "min_mfma_flops=1")
    ks = [x for x in hip.code.kernels() if x["kind"] == "mfma"]
    if not ks and nodes[out].prec == "bfloat16":
        # a sum that one thread runs, rounded after every addition: left alone, and the oracle's bits
        oracle = OracleRun(r, init)
        hip.step(); oracle.step()
        assert np.array_equal(hip.get(nodes[out]).ravel(), np.asarray(oracle.get(nodes[out])).ravel())
        return hip.close()
    assert ks and all("_kernel_any" in x["name"] for x in ks), hip.code.kernels()
    hip.step()
    f = {name: W.to_float(init[n.id], n.prec).astype(np.float64) for name, n in nodes.items()}
    ref = want(f) + (f[out] if accumulate else 0.0)
    got = W.to_float(hip.get(nodes[out]), nodes[out].prec).astype(np.float64)
    err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    tol = 2.0 ** -8 if nodes[out].prec == "bfloat16" else 2e-6 * max(1.0, np.sqrt(k) / 8)
    assert err <= tol, (err, tol, ks[0]["name"])
    hip.close()


def _product(M, N, K, a_prec, b_prec, c_prec, a_kc, b_kc, accumulate, batch=0, seed=0, direct=None):
    r, A, B, C = _routine(M, N, K, a_prec, b_prec, c_prec, a_kc, b_kc, accumulate, batch)
    t = lambda x, kc: x if kc else np.swapaxes(x, -1, -2)
    if direct is not None:
        names = [k["name"] for k in backend.compile(r, "min_mfma_flops=1").kernels() if k["kind"] == "mfma"]
        assert len(names) == 1 and ("_any_direct<" in names[0]) == direct, names
    _run(r, dict(a=A, b=B, c=C), "c", lambda f: t(f["a"], a_kc) @ np.swapaxes(t(f["b"], b_kc), -1, -2), accumulate, K, seed)


@pytest.mark.parametrize("layout", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("precs", [("bfloat16", "bfloat16", "single"), ("bfloat16", "bfloat16", "bfloat16"), ("single", "bfloat16", "single"),
                                   ("bfloat16", "single", "bfloat16"), ("single", "single", "single")])
def test_odd_extents(layout, precs):
    for seed, (M, N, K) in enumerate(((65, 63, 67), (17, 9, 9), (129, 131, 31), (63, 65, 257))):
        _product(M, N, K, *precs, *layout, accumulate=seed % 2 == 0, seed=seed)


@pytest.mark.parametrize("layout", [(True, True), (False, False), (True, False)])
@pytest.mark.parametrize("prec", ["bfloat16", "single"])
def test_large_tiles_splits_and_batches(layout, prec):
    _product(2049, 4099, 130, prec, prec, "single", *layout, accumulate=False, seed=1)      # 128 x 128 tiles
    _product(33, 70, 4099, prec, prec, "single", *layout, accumulate=True, seed=2)          # K split
    _product(71, 19, 2051, prec, prec, "bfloat16", *layout, accumulate=True, seed=3)
    _product(99, 37, 45, prec, prec, "single", *layout, accumulate=False, batch=11, seed=4)


@pytest.mark.parametrize("prec", ["bfloat16", "single"])
@pytest.mark.parametrize("shape", [dict(b=3, oh=9, ow=7, ic=5, oc=17), dict(b=2, oh=16, ow=12, ic=8, oc=24), dict(b=5, oh=6, ow=11, ic=3, oc=19)])
@pytest.mark.parametrize("stride,ksz", [(1, 3), (2, 3), (3, 2)])
def test_convolution_windows(stride, ksz, shape, prec):
    # y += x * w and w_grad += y_grad * x: rows and sums of several loop symbols that do not merge
    full, n = _conv(stride, ksz, prec, **shape)
    nests = [s for s in full.body if not isinstance(s, L.ZeroOut)]
    names = ("x", "w", "y", "dy", "dw")
    n["y"].prec = n["dw"].prec = "single"
    nodes = {k: n[k] for k in names}
    oh, ow = shape["oh"], shape["ow"]
    window = lambda x, k1, k2: x[:, k1:k1 + stride * (oh - 1) + 1:stride, k2:k2 + stride * (ow - 1) + 1:stride, :]

    def fwd(f):
        return sum(np.einsum("bhwi,ci->bhwc", window(f["x"], k1, k2), f["w"][:, k1, k2, :]) for k1 in range(ksz) for k2 in range(ksz))

    def dw(f):
        out = np.zeros(n["dw"].dims)
        for k1 in range(ksz):
            for k2 in range(ksz):
                out[:, k1, k2, :] = np.einsum("bhwc,bhwi->ci", f["dy"], window(f["x"], k1, k2))
        return out

    ins = lambda *k: {x: nodes[x] for x in k}
    _run(L.Routine("conv_fwd", [nests[0]]), ins("x", "w", "y"), "y", fwd, True, ksz * ksz * shape["ic"])
    _run(L.Routine("conv_dw", [nests[2]]), ins("x", "dy", "dw"), "dw", dw, True, shape["b"] * oh * ow)


def test_slices_at_any_offset():
    # the operands are slices that start at odd elements of larger tensors
    L.reset_symbols(0)
    M, N, K = 70, 41, 53
    a = L.Node(1, "a", "bfloat16", (M + 1, K + 3)); b = L.Node(2, "b", "bfloat16", (K + 1, N + 2)); c = L.Node(3, "c", "single", (M, N + 1))
    m, n, k = (L.fresh_symbol() for _ in range(3))
    at = lambda s, o: L.Affine(((1, s),), o)
    ci = (L.It(m), at(n, 1))
    body = L.Set(c, ci, L.Ternop("fma", L.Get(a, (at(m, 1), at(k, 3))), L.Get(b, (at(k, 1), at(n, 1))), L.Get(c, ci)))
    for sym, ext in ((k, K), (n, N), (m, M)):
        body = L.For(sym, 0, ext - 1, [body])

    def want(f):
        out = np.zeros(c.dims)
        out[:, 1:] = f["a"][1:, 3:] @ f["b"][1:, 1:N + 1]
        return out
    _run(L.Routine("slices", [body]), dict(a=a, b=b, c=c), "c", want, True, K)


@pytest.mark.parametrize("prec", ["bfloat16", "single"])
@pytest.mark.parametrize("shape", [dict(b=3, oh=9, ow=7, ic=5, oc=16), dict(b=2, oh=16, ow=12, ic=40, oc=24), dict(b=1, oh=6, ow=11, ic=3, oc=9)])
@pytest.mark.parametrize("stride,ksz", [(1, 3), (2, 3), (2, 5), (3, 4)])
@pytest.mark.parametrize("zeroed", [True, False])
def test_overlapping_windows_are_gathered(stride, ksz, shape, prec, zeroed):
    # x_grad[stride * o + k] += y_grad[o] * w[k]: turned round into a sum over the taps that reach a position
    full, n = _conv(stride, ksz, prec, **shape)
    n["dx"].prec = "single"
    r = L.Routine("conv_dx", ([L.ZeroOut(n["dx"])] if zeroed else []) + [[s for s in full.body if not isinstance(s, L.ZeroOut)][1]])
    rng = np.random.default_rng(stride)
    init = {n[k].id: _values(rng, n[k]) for k in ("w", "dy", "dx")}
    hip = HipRun(r, init, "min_mfma_flops=1")
    assert [k["kind"] for k in hip.code.kernels()] == ["generated"] and "ocn_any_tile<" in hip.code.source().split('extern "C"')[1]
    hip.step()
    w, dy = (W.to_float(init[n[k].id], prec).astype(np.float64) for k in ("w", "dy"))
    want = np.zeros(n["dx"].dims) if zeroed else init[n["dx"].id].astype(np.float64)
    oh, ow = shape["oh"], shape["ow"]
    for k1 in range(ksz):
        for k2 in range(ksz):
            want[:, k1:k1 + stride * (oh - 1) + 1:stride, k2:k2 + stride * (ow - 1) + 1:stride, :] += np.einsum("bhwc,ci->bhwi", dy, w[:, k1, k2, :])
    assert np.max(np.abs(hip.get(n["dx"]) - want)) <= 4e-6 * np.max(np.abs(want))
    hip.close()


@pytest.mark.parametrize("prec", ["bfloat16", "single"])
@pytest.mark.parametrize("taps,stride,ic", [((3, 3), (2, 1), 32), ((1, 3), (2, 2), 32), ((3, 1), (2, 2), 40), ((2, 3), (3, 2), 5), ((1, 4), (4, 3), 5)])
@pytest.mark.parametrize("taps_first", [True, False])
@pytest.mark.parametrize("zeroed", [True, False])
def test_windows_of_any_taps_steps_and_weight_layout(taps, stride, ic, prec, taps_first, zeroed):
    # steps that some residues of an axis have no tap for: those positions are zeros, or stay as they were
    r, nodes, want = input_gradient(taps, stride, prec, taps_first, b=3, oh=9, ow=7, ic=ic, oc=ic, zeroed=zeroed)
    rng = np.random.default_rng(ic)
    init = {n.id: _values(rng, n) for n in nodes}
    hip = HipRun(r, init, "min_mfma_flops=1")
    assert "ocn_any_tile<" in hip.code.source().split('extern "C"')[1]
    hip.step()
    ref = want({n.ident: W.to_float(init[n.id], n.prec).astype(np.float64) for n in nodes})
    assert np.max(np.abs(hip.get(nodes[2]) - ref)) <= 4e-6 * np.max(np.abs(ref))
    hip.close()


@pytest.mark.parametrize("prec", ["bfloat16", "single"])
@pytest.mark.parametrize("taps,stride,ic", [((3, 3), (1, 1), 33), ((3, 2), (2, 1), 40), ((5, 3), (2, 2), 5), ((3, 3), (1, 1), 64)])
@pytest.mark.parametrize("zeroed", [True, False])
def test_a_weight_counts_only_where_its_tap_reaches(taps, stride, ic, prec, zeroed):
    r, nodes, want = input_gradient(taps, stride, prec, not zeroed, oh=9, ow=7, ic=ic, oc=16, zeroed=zeroed)
    init, values = non_finite(nodes, ic)
    hip = HipRun(r, {n.id: init[n.ident] for n in nodes}, "min_mfma_flops=1")
    hip.step()
    with np.errstate(invalid="ignore"):
        ref = want(values)
    _same_numbers(hip.get(nodes[2]), ref, 4e-6)
    hip.close()


@pytest.mark.parametrize("late", [False, True])
def test_a_product_reads_what_the_window_gather_left(late):
    r, n = gathered_then_multiplied(late)
    rng = np.random.default_rng(5)
    init = {x.id: _values(rng, x) for x in n.values()}
    hip = HipRun(r, init, "min_mfma_flops=1")
    hip.step()
    f = {k: W.to_float(init[x.id], x.prec).astype(np.float64) for k, x in n.items()}
    rounded = lambda x: W.to_float(W.as_prec(x.astype(np.float32), "bfloat16"), "bfloat16").astype(np.float64)
    times_h = lambda x: np.einsum("bpg,bpi->gi", f["h"], rounded(x))
    dx = f["r"].copy()
    for k in range(3):
        dx[:, k:k + 16] += np.einsum("boc,ci->boi", f["dy"], f["w"][:, k])
    for name, want in (("dx", dx), ("out", times_h(hip.get(n["dx"]).astype(np.float64)))) + ((("first", times_h(f["r"])),) if late else ()):
        assert np.max(np.abs(hip.get(n[name]) - want)) <= 4e-6 * np.max(np.abs(want)), name
    hip.close()


@pytest.mark.parametrize("shape", [(3, 72, 40, 72), (5, 136, 72, 200), (2, 24, 200, 64)])
@pytest.mark.parametrize("one_statement", [False, True])
def test_bias_and_relu_of_every_batch_entry(shape, one_statement):
    # y[z, b, o] := (the inlined product) + bias[o]; relu(y), stored by the contraction itself, per batch entry
    from ocannl_amd.frontend import Graph, make_routine
    Z, M, N, K = shape
    L.reset_symbols(0)
    g = Graph("bfloat16", "single")
    x = g.input("x", ("z", "b", "i"), (Z, M, K)); w = g.param("w", ("z", "o", "i"), (Z, N, K)); bias = g.param("bias", ("o",), (N,))
    y = g.add(g.einsum(w, x, ("z", "b", "o"), ident="wx"), bias, ("z", "b", "o"), ident="y")
    relu = g.unary("relu", y, ident="relu")
    r = make_routine(g, "layers", g.forward(relu), outputs=[relu.value] if one_statement else [y.value, relu.value], **({"inline": "visits"} if one_statement else {}))
    rng = np.random.default_rng(M)
    init = {t.value.id: W.as_prec((rng.standard_normal(t.value.dims) / np.sqrt(K if t is w else 1)).astype(np.float32), "bfloat16") for t in (x, w, bias)}
    folded, apart = HipRun(r, init, "min_mfma_flops=1"), HipRun(r, init, "min_mfma_flops=1;epilogues=0;fused=0")
    assert [k["name"].split("<")[0] for k in folded.code.kernels()] == ["gemm_bf16_kernel_any" + ("_direct" if K > 64 else "")] and len(apart.code.kernels()) > 1
    folded.step(); apart.step()
    f = {t: W.to_float(init[t.value.id], "bfloat16").astype(np.float64) for t in (x, w, bias)}
    want = np.einsum("zbi,zoi->zbo", f[x], f[w]) + f[bias]
    for t, ref in ([] if one_statement else [(y, want)]) + [(relu, np.maximum(want, 0))]:
        got = folded.get(t.value)
        assert np.array_equal(got, apart.get(t.value)), t.value.ident
        # (the product is rounded, and its sum with the bias again: 2^-9 of either, of at most the largest)
        assert np.max(np.abs(W.to_float(got, "bfloat16") - ref)) <= 2.0 ** -7 * np.max(np.abs(want))
    folded.close(); apart.close()


def _forms(kernels):
    return [k["name"].split("<")[0] for k in kernels if k["kind"] == "mfma"]


@pytest.mark.parametrize("layout", [(True, True), (False, False), (True, False), (False, True)])
@pytest.mark.parametrize("precs", [("bfloat16", "bfloat16", "single"), ("single", "single", "single"), ("single", "bfloat16", "single"), ("bfloat16", "single", "single")])
@pytest.mark.parametrize("M,N,K,batch", [(40, 30, 66, 0), (33, 18, 97, 5), (16, 8, 127, 0), (70, 66, 200, 7), (34, 130, 3100, 0)])
def test_few_tiles_share_k_among_wavefronts(M, N, K, batch, precs, layout):
    # one step of K for some wavefronts and none for others, a partial step, rows past the end, batch entries, K splits
    # (rows of bf16 at odd elements, and long sums of two k-contiguous bf16 operands, go to staged tiles)
    bf16 = precs[:2] == ("bfloat16", "bfloat16")
    staged = any(p == "bfloat16" and kc and K % 2 for p, kc in zip(precs, layout)) or (bf16 and all(layout) and K > 256)
    _product(M, N, K, *precs, *layout, accumulate=K % 2 == 0, batch=batch, seed=K, direct=not staged)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("precs", [("bfloat16", "bfloat16", "bfloat16"), ("single", "single", "bfloat16"), ("single", "bfloat16", "bfloat16")])
def test_few_tiles_store_bf16(precs, accumulate):
    _product(71, 66, 202, *precs, True, False, accumulate=accumulate, seed=7, direct=True)


@pytest.mark.parametrize("layout", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("precs", [("bfloat16", "bfloat16"), ("single", "bfloat16"), ("bfloat16", "single")])
@pytest.mark.parametrize("K", [73, 97, 131, 189])
def test_few_tiles_with_an_odd_end_of_k(K, precs, layout):
    # sums over the first K columns of rows of K + 1, so that bf16 rows start at even elements and the last chunk is shifted
    # by an odd number of halves
    M, N = 70, 66
    L.reset_symbols(0)
    a = L.Node(1, "a", precs[0], (M, K + 1) if layout[0] else (K + 1, M)); b = L.Node(2, "b", precs[1], (N, K + 1) if layout[1] else (K + 1, N))
    c = L.Node(3, "c", "single", (M, N))
    m, n, k = (L.fresh_symbol() for _ in range(3))
    at = lambda r, kc: (L.It(r), L.It(k)) if kc else (L.It(k), L.It(r))
    body = L.Set(c, (L.It(m), L.It(n)), L.Ternop("fma", L.Get(a, at(m, layout[0])), L.Get(b, at(n, layout[1])), L.Get(c, (L.It(m), L.It(n)))))
    for sym, ext in ((k, K), (n, N), (m, M)):
        body = L.For(sym, 0, ext - 1, [body])
    r = L.Routine("odd_end", [L.ZeroOut(c), body])
    name, = [x["name"] for x in backend.compile(r, "min_mfma_flops=1").kernels() if x["kind"] == "mfma"]
    assert "_any_direct<" in name, name
    t = lambda x, kc: x[:, :K] if kc else x[:K].T
    _run(r, dict(a=a, b=b, c=c), "c", lambda f: t(f["a"], layout[0]) @ t(f["b"], layout[1]).T, False, K, K)


@pytest.mark.parametrize("layout", [(True, True), (False, False), (True, False)])
@pytest.mark.parametrize("precs,form", [(("single", "single"), "f32_kernel_any<"), (("single", "single"), "f32_kernel_any_direct<"), (("single", "single"), "f32_kernel<"),
                                        (("single", "bfloat16"), "f32_kernel_any<"), (("single", "bfloat16"), "f32_kernel_any_direct<"),
                                        (("bfloat16", "single"), "f32_kernel_any<"), (("bfloat16", "single"), "f32_kernel_any_direct<")])
@pytest.mark.parametrize("sa,sb", [(-142, 40), (-130, 20), (-60, -60), (30, -128), (0, 0)])
def test_single_products_in_bf16_parts(sa, sb, precs, form, layout):
    """One non-zero value in a row of A, of around 2^sa (subnormal ones too), so that a cell is one product: as exact as
    an fp32 product, whatever the parts' exponents."""
    M, N, K = (70, 66, 132) if "direct" in form else (1032, 1100, 152) if form.endswith("kernel<") else (1031, 1099, 151)
    r, A, B, C = _routine(M, N, K, *precs, "single", *layout, False)
    rng = np.random.default_rng(6)
    a, b = np.zeros((M, K), np.float32), np.ldexp(rng.standard_normal((N, K)), sb).astype(np.float32)
    a[np.arange(M), rng.integers(K, size=M)] = np.ldexp(rng.standard_normal(M), sa).astype(np.float32)
    t = lambda x, kc, p: W.as_prec(np.ascontiguousarray(x if kc else x.T), p)
    hip = HipRun(r, {1: t(a, layout[0], precs[0]), 2: t(b, layout[1], precs[1])}, "min_mfma_flops=1;bf16_copies=0" + (";any=0" if form.endswith("kernel<") else ""))
    assert form in hip.code.kernels()[-1]["name"], hip.code.kernels()
    hip.step()
    got = hip.get(C).astype(np.float64)
    hip.close()
    f = lambda x, p: W.to_float(W.as_prec(x, p), p).astype(np.float64)
    want = f(a, precs[0]) @ f(b, precs[1]).T
    # the six part products (or three) are added one after the other, each sum off by less than 2^-23 of the result; the
    # three left out are below 2^-24 of it together; the result itself may be subnormal
    assert np.all(np.abs(got - want) <= 7 * 2.0 ** -23 * np.abs(want) + 2.0 ** -149)


@pytest.mark.parametrize("layout", [(True, True), (False, False), (True, False)])
@pytest.mark.parametrize("precs", [("single", "single"), ("single", "bfloat16"), ("bfloat16", "single")])
@pytest.mark.parametrize("M,N,K", [(70, 66, 131), (1031, 1099, 150), (30, 9000, 150), (2049, 4099, 135)])
@pytest.mark.parametrize("what", ["tiny", "special"])
def test_values_that_three_bf16_parts_do_not_cover(M, N, K, precs, layout, what):
    """Values below 2^-102, infinities, NaN and values above the largest bf16 give what fp32 products give."""
    if (M > 2000 and precs != ("single", "single")) or (M == 30 and "bfloat16" in precs):
        pytest.skip("tiles of fp32 operands only")
    r, A, B, C = _routine(M, N, K, *precs, "single", *layout, False)
    rng = np.random.default_rng(4)
    a, b = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((N, K)).astype(np.float32)
    if what == "tiny":
        x, y = (a, b) if precs[0] == "single" else (b, a)
        x[: len(x) // 2] *= np.float32(2.0 ** -118)
        y *= np.float32(2.0 ** 30)
        y[:, K // 2:] = 1.0                      # (whose mid and lo parts are zero)
    else:
        b[:, :4] = 1.0
        a[3, 1], a[M - 1, 0], a[M // 2, 2], b[N - 2, K - 1] = np.inf, -np.inf, np.nan, np.float32(3.3e38)
        a[:, K - 1] = rng.choice(np.float32([0.5, 0.25]), M)
    a, b = (W.to_float(W.as_prec(x, p), p) for x, p in ((a, precs[0]), (b, precs[1])))
    t = lambda x, kc, p: W.as_prec(np.ascontiguousarray(x if kc else x.T), p)
    hip = HipRun(r, {1: t(a, layout[0], precs[0]), 2: t(b, layout[1], precs[1])}, "min_mfma_flops=1;bf16_copies=0")
    assert all("_kernel_any" in f for f in _forms(hip.code.kernels())), hip.code.kernels()
    hip.step()
    got = hip.get(C).astype(np.float64)
    hip.close()
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64).T
        size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T
    fine = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)])
    # K roundings of fp32, each of half a unit of a partial sum that is no larger than `size`
    assert (np.abs(got[fine] - want[fine]) / size[fine]).max() <= K * 2.0 ** -24
