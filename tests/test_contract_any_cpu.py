"""What the planner hands to the contraction tile for any shape, and what that tile reads; no GPU needed."""
import os
import re
import subprocess

import numpy as np
import pytest

from ocannl_amd import backend as B
from ocannl_amd import llir as L
from ocannl_amd import workloads as W


def _product(M, N, K, prec="single", a_kc=True, b_kc=True):
    L.reset_symbols(0)
    a = L.Node(1, "a", prec, (M, K) if a_kc else (K, M)); b = L.Node(2, "b", prec, (N, K) if b_kc else (K, N)); c = L.Node(3, "c", "single", (M, N))
    m, n, k = (L.fresh_symbol() for _ in range(3))
    at = lambda r, s, kc: (L.It(r), L.It(s)) if kc else (L.It(s), L.It(r))
    body = L.Set(c, at(m, n, True), L.Ternop("fma", L.Get(a, at(m, k, a_kc)), L.Get(b, at(n, k, b_kc)), L.Get(c, at(m, n, True))))
    for sym, ext in ((k, K), (n, N), (m, M)):
        body = L.For(sym, 0, ext - 1, [body])
    return L.Routine("product", [L.ZeroOut(c), body])


def _matrix_kernels(r):
    return [k["name"] for k in B.compile(r, "min_mfma_flops=1").kernels() if k["kind"] == "mfma"]


@pytest.mark.parametrize("layout", [(True, True), (False, False)])
@pytest.mark.parametrize("prec", ["single", "bfloat16"])
def test_operands_beyond_32_bit_offsets_keep_the_64_bit_kernels(layout, prec):
    # the tile's element offsets within one batch entry are ints: 2^21 * 264 elements fit, 2^23 * 264 do not
    assert "kernel_any<" in _matrix_kernels(_product(264, 264, 1 << 21, prec, *layout))[0]
    name, = _matrix_kernels(_product(264, 264, 1 << 23, prec, *layout))
    assert "kernel_any<" not in name


@pytest.mark.parametrize("prec", ["single", "bfloat16"])
@pytest.mark.parametrize("shape,layout,small", [((1000, 1000, 1024), (False, False), True), ((1000, 1000, 8192), (False, False), False),
                                                ((1000, 1000, 8192), (True, True), False), ((264, 264, 8192), (False, False), True),
                                                ((2040, 1528, 8192), (True, True), True), ((1784, 776, 8192), (False, False), False)])
def test_small_tiles_where_they_go_through_less(shape, layout, small, prec):
    # a long sum over few tiles: the register-staged kernels split it further and re-read less
    name, = _matrix_kernels(_product(*shape, prec, *layout))
    assert ("kernel_any<64, 64" in name) == small


@pytest.mark.parametrize("local_mib,small", [(0, False), (8, True), (31, True), (40, False)])
def test_a_workspace_does_not_take_a_routine_beyond_the_static_scratch(local_mib, small):
    # 1000 x 1000 x 8192 staged: eight splits, 30.5 of 32 MiB; beside local tensors that leave less the small tile, which
    # needs none, keeps the routine runnable without an allocation (beyond 32 MiB it is not, either way)
    r = _product(1000, 1000, 8192, "single", False, False)
    if local_mib:
        i, n = L.fresh_symbol(), local_mib << 18
        src, local, out = L.Node(4, "src", "single", (n,)), L.Node(5, "local", "single", (n,), mode="local"), L.Node(6, "out", "single", (n,))
        at = (L.It(i),)
        copy = lambda d, s: L.For(i, 0, n - 1, [L.Set(d, at, L.Unop("neg", L.Get(s, at)))])
        r.body.extend([copy(local, src), copy(out, local)])
    name, = _matrix_kernels(r)
    assert ("kernel_any<64, 64" in name) == small


def _products(M, N, K, precs, a_kc, b_kc, batch=1, members=1):
    L.reset_symbols(0)
    z, m, n, k = (L.fresh_symbol() for _ in range(4))
    at = lambda r, s, kc: (L.It(z),) + ((L.It(r), L.It(s)) if kc else (L.It(s), L.It(r)))
    a, body = L.Node(1, "a", precs[0], (batch, M, K) if a_kc else (batch, K, M)), []
    for g in range(members):
        b = L.Node(2 + 2 * g, f"b{g}", precs[1], (batch, N, K) if b_kc else (batch, K, N)); c = L.Node(3 + 2 * g, f"c{g}", "single", (batch, M, N))
        nest = L.Set(c, at(m, n, True), L.Ternop("fma", L.Get(a, at(m, k, a_kc)), L.Get(b, at(n, k, b_kc)), L.Get(c, at(m, n, True))))
        for sym, ext in ((k, K), (n, N), (m, M), (z, batch)):
            nest = L.For(sym, 0, ext - 1, [nest])
        body += [L.ZeroOut(c), nest]
    return L.Routine("products", body)


F, H = "single", "bfloat16"


@pytest.mark.parametrize("M,N,K,precs,layout,batch,members,direct", [
    # one tile a compute unit, and one more; long sums in fp32, unsplit, two splits, four
    (511, 511, 1000, (F, F), (True, True), 1, 1, True), (545, 481, 1000, (F, F), (True, True), 1, 1, False), (511, 511, 1800, (F, F), (True, True), 1, 1, True),
    (511, 511, 1801, (F, F), (True, True), 1, 1, False), (511, 511, 2048, (F, F), (True, False), 1, 1, True), (511, 511, 2049, (F, F), (True, False), 1, 1, False),
    (255, 511, 3071, (F, F), (True, True), 1, 1, True), (255, 511, 3072, (F, F), (True, True), 1, 1, False), (255, 255, 4096, (F, F), (True, True), 1, 1, True),
    # up to two a unit, with a row-contiguous operand
    (511, 1023, 1536, (F, F), (True, False), 1, 1, True), (511, 1023, 1537, (F, F), (True, False), 1, 1, False), (511, 1055, 512, (F, F), (True, False), 1, 1, False),
    (511, 1023, 96, (F, F), (True, False), 1, 1, True), (511, 1023, 128, (F, F), (True, False), 1, 1, False), (511, 1023, 128, (F, F), (False, False), 1, 1, True),
    # bf16
    (511, 511, 3071, (H, H), (False, False), 1, 1, True), (511, 511, 3072, (H, H), (False, False), 1, 1, False), (255, 511, 4096, (H, H), (False, False), 1, 1, True),
    (511, 545, 512, (H, H), (False, False), 1, 1, False), (300, 300, 160, (H, H), (True, True), 1, 1, True), (300, 300, 128, (H, H), (True, True), 1, 1, False),
    (300, 300, 256, (H, H), (True, True), 1, 1, True), (300, 300, 260, (H, H), (True, True), 1, 1, False), (301, 301, 510, (H, F), (True, True), 1, 1, True),
    # batches of one tile, which is mostly padding of a staged one; groups go by all of their tiles
    (31, 31, 4000, (F, F), (True, True), 200, 1, True), (63, 31, 4000, (F, F), (True, True), 128, 1, True), (95, 31, 4000, (F, F), (True, True), 60, 1, False),
    (256, 256, 4096, (F, F), (True, True), 1, 1, True), (256, 256, 4096, (F, F), (True, True), 1, 4, False), (256, 512, 2048, (F, F), (True, True), 1, 1, True),
    (256, 512, 2048, (F, F), (True, True), 1, 2, False), (512, 256, 512, (F, F), (True, True), 1, 4, True), (512, 256, 520, (F, F), (True, True), 1, 4, False)])
def test_few_tiles_share_k_where_that_is_measured_to_be_faster(M, N, K, precs, layout, batch, members, direct):
    code = B.compile(_products(M, N, K, precs, *layout, batch, members), "min_mfma_flops=1;bf16_copies=0")
    name, = {k["name"] for k in code.kernels() if k["kind"] == "mfma"}
    assert ("_any_direct<" in name) == direct, name
    assert direct or "kernel_any<" in name, name


def test_sums_of_more_terms_than_32_bits_count_are_left_alone():
    # k in two digits over operands of few elements: x[i + j] * w[i + j], 2^31 terms and more
    def names(I, J):
        L.reset_symbols(0)
        x = L.Node(1, "x", "single", (24, I + J)); w = L.Node(2, "w", "single", (24, I + J)); c = L.Node(3, "c", "single", (24, 24))
        m, n, i, j = (L.fresh_symbol() for _ in range(4))
        at = lambda r: (L.It(r), L.Affine(((1, i), (1, j)), 0))
        body = L.Set(c, (L.It(m), L.It(n)), L.Ternop("fma", L.Get(x, at(m)), L.Get(w, at(n)), L.Get(c, (L.It(m), L.It(n)))))
        for sym, ext in ((j, J), (i, I), (n, 24), (m, 24)):
            body = L.For(sym, 0, ext - 1, [body])
        return _matrix_kernels(L.Routine("terms", [L.ZeroOut(c), body]))
    assert "kernel_any<" in names(300, 200)[0]
    assert not names(1 << 17, 1 << 14)


def test_a_window_step_beyond_its_axis_is_not_gathered():
    # one position with a step of 2^20: the gather would launch a tile for each residue of the step
    def source(step, oh, ic=2):
        L.reset_symbols(0)
        dy = L.Node(1, "dy", "single", (64, oh, 32)); w = L.Node(2, "w", "single", (32, 3, ic)); dx = L.Node(3, "dx", "single", (64, 16, ic))
        b, o, k, c, i = (L.fresh_symbol() for _ in range(5))
        at = (L.It(b), L.Affine(((step, o), (1, k)), 0), L.It(i))
        body = L.Set(dx, at, L.Ternop("fma", L.Get(dy, (L.It(b), L.It(o), L.It(c))), L.Get(w, (L.It(c), L.It(k), L.It(i))), L.Get(dx, at)))
        for sym, ext in ((i, ic), (k, 3), (c, 32), (o, oh), (b, 64)):
            body = L.For(sym, 0, ext - 1, [body])
        return B.compile(L.Routine("window", [body]), "min_mfma_flops=1").source().split('extern "C"')[1]
    assert "ocn_any_tile<" in source(2, 5)
    assert "ocn_any_tile<" not in source(1 << 20, 1)


def gathered_then_multiplied(late):
    """dx := r; dx += windows of dy * w; out := h^T dx, h in bf16 (so that the product reads dx rounded); with `late` the
    product also runs ahead of the windows, into first."""
    L.reset_symbols(0)
    b, o, taps, ic, g = 4, 16, 3, 32, 32
    p = o + taps - 1
    w = L.Node(1, "w", "bfloat16", (ic, taps, ic)); dy = L.Node(2, "dy", "bfloat16", (b, o, ic)); r = L.Node(3, "r", "single", (b, p, ic))
    h = L.Node(4, "h", "bfloat16", (b, p, g)); dx = L.Node(5, "dx", "single", (b, p, ic)); out = L.Node(6, "out", "single", (g, ic)); first = L.Node(7, "first", "single", (g, ic))

    def nest(exts, stmt):
        syms = [L.fresh_symbol() for _ in exts]
        body = [stmt(*(L.It(s) for s in syms), *syms)]
        for s, e in reversed(list(zip(syms, exts))):
            body = [L.For(s, 0, e - 1, body)]
        return body
    product = lambda c: [L.ZeroOut(c)] + nest((g, ic, b, p), lambda m, n, k, l, *_: L.Set(c, (m, n), L.Ternop("fma", L.Get(h, (k, l, m)), L.Get(dx, (k, l, n)), L.Get(c, (m, n)))))
    at = lambda syms: (L.It(syms[0]), L.Affine(((1, syms[1]), (1, syms[2])), 0), L.It(syms[4]))
    body = nest((b, p, ic), lambda i, j, k, *_: L.Set(dx, (i, j, k), L.Get(r, (i, j, k)))) + (product(first) if late else [])
    body += nest((b, o, taps, ic, ic), lambda bb, oo, k, c, i, *s: L.Set(dx, at(s), L.Ternop("fma", L.Get(dy, (bb, oo, c)), L.Get(w, (c, k, i)), L.Get(dx, at(s)))))
    return L.Routine("gathered", body + product(out)), dict(w=w, dy=dy, r=r, h=h, dx=dx, out=out, **({"first": first} if late else {}))


@pytest.mark.parametrize("late", [False, True])
def test_a_bf16_copy_is_made_after_the_window_gather_that_writes_its_tensor(late):
    # (the copy that generated stores keep in step: the gather stores the tensor alone)
    r, _ = gathered_then_multiplied(late)
    code = B.compile(r, "min_mfma_flops=1")
    kernels = re.findall(r'extern "C" __global__ void[^(]*\(256\) \w+\(([^)]*)\) \{(.*?)\n\}\n', code.source(), re.S)
    gather = [i for i, (_, body) in enumerate(kernels) if "ocn_any_tile<" in body]
    assert len(gather) == 1 and any("bf" in params and "_dx" in params for params, _ in kernels[gather[0] + 1:])


# ---- the window gather, run on the host --------------------------------------------------------------

CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")


def _on_the_host(tmp_path, code, values):
    """The one kernel of `code` in a host program (host_workgroup.h): the tensors by name, as it leaves them, and under
    "f32_products" the fp32 matrix instructions it went through."""
    source = code.source()
    tile, kernel = source[source.index("template <bool C, typename A"):], source[source.index('extern "C" __global__'):]
    name, params = re.match(r'extern "C" __global__ void __launch_bounds__\(256\) (\w+)\(([^)]*)\)', kernel).groups()
    types, names = zip(*(p.replace("__restrict__", "").split("*") for p in params.split(",")))
    names = [n.strip() for n in names]
    call = ", ".join(f"({t.strip()}*)p[{i}]" for i, t in enumerate(types))
    (tmp_path / "kernel.cpp").write_text(f'#include "host_workgroup.h"\n{tile}\nvoid host_kernel(void** p) {{ {name}({call}); }}\n')
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-ffp-contract=off", "-I", os.path.dirname(os.path.abspath(__file__)), "kernel.cpp", "-o", "kernel"],
                   cwd=tmp_path, check=True)
    arrays = [np.ascontiguousarray(values[n]) for n in names]
    (tmp_path / "tensors").write_bytes(b"".join(a.tobytes() for a in arrays))
    blocks = 8 * int(re.search(r"blockIdx.x % 8u\) \* (\d+)", kernel).group(1))
    p = subprocess.run([tmp_path / "kernel", str(blocks), tmp_path / "tensors"] + [str(a.nbytes) for a in arrays], check=True, timeout=120, stdout=subprocess.PIPE)
    raw, out, at = (tmp_path / "tensors").read_bytes(), {"f32_products": int(p.stdout)}, 0
    for n, a in zip(names, arrays):
        out[n] = np.frombuffer(raw, a.dtype, a.size, at).reshape(a.shape)
        at += a.nbytes
    return out


def input_gradient(taps, stride, prec, taps_first, b=2, oh=5, ow=4, ic=32, oc=32, zeroed=True):
    """x_grad[b, s1 * o1 + k1, s2 * o2 + k2, i] += y_grad[b, o1, o2, c] * w[c, k1, k2, i], the weights stored in that
    order or as [k1, k2, i, c]; and the same from float64 values by name, the taps that reach a position and no others."""
    L.reset_symbols(0)
    (kh, kw), (s1, s2) = taps, stride
    w = L.Node(1, "w", prec, (kh, kw, ic, oc) if taps_first else (oc, kh, kw, ic)); dy = L.Node(2, "dy", prec, (b, oh, ow, oc))
    dx = L.Node(3, "dx", "single", (b, s1 * (oh - 1) + kh, s2 * (ow - 1) + kw, ic))
    bb, o1, o2, c, k1, k2, i = syms = [L.fresh_symbol() for _ in range(7)]
    at = (L.It(bb), L.Affine(((s1, o1), (1, k1)), 0), L.Affine(((s2, o2), (1, k2)), 0), L.It(i))
    wi = (L.It(k1), L.It(k2), L.It(i), L.It(c)) if taps_first else (L.It(c), L.It(k1), L.It(k2), L.It(i))
    body = [L.Set(dx, at, L.Ternop("fma", L.Get(dy, (L.It(bb), L.It(o1), L.It(o2), L.It(c))), L.Get(w, wi), L.Get(dx, at)))]
    for sym, ext in reversed(list(zip(syms, (b, oh, ow, oc, kh, kw, ic)))):
        body = [L.For(sym, 0, ext - 1, body)]

    def want(f):
        out = np.zeros(dx.dims) if zeroed else f["dx"].copy()
        weights = f["w"].transpose(3, 0, 1, 2) if taps_first else f["w"]
        for r in range(kh):
            for s in range(kw):
                at = out[:, r:r + s1 * (oh - 1) + 1:s1, s:s + s2 * (ow - 1) + 1:s2, :]
                for k in range(oc):   # (term by term: a library product may move a NaN where no term has one)
                    at += f["dy"][..., k, None] * weights[k, r, s, :]
        return out
    return L.Routine("dx", ([L.ZeroOut(dx)] if zeroed else []) + body), (w, dy, dx), want


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm compiler")
@pytest.mark.parametrize("prec", ["single", "bfloat16"])
@pytest.mark.parametrize("taps,stride,ic", [((3, 3), (2, 1), 32), ((1, 3), (2, 2), 32), ((3, 1), (2, 2), 40), ((2, 3), (3, 2), 5), ((1, 4), (4, 3), 5)])
def test_window_gathers_stay_inside_their_operands(taps, stride, ic, prec, tmp_path):
    # a residue of the step that no tap has reads no weights: behind them lies a page that may not be touched
    for taps_first in (True, False):
        r, nodes, want = input_gradient(taps, stride, prec, taps_first, ic=ic, oc=ic, zeroed=taps_first)
        code = B.compile(r, "min_mfma_flops=1")
        assert "ocn_any_tile<" in code.source().split('extern "C"')[1]
        rng = np.random.default_rng(ic)
        init = {n.ident: W.as_prec(rng.standard_normal(n.dims).astype(np.float32), n.prec) for n in nodes}
        ref = want({n.ident: W.to_float(init[n.ident], n.prec).astype(np.float64) for n in nodes})
        # fp32 sums of at most 9 x 40 terms: their rounding is below 2^-24 a term, of the size of the largest result
        assert np.max(np.abs(_on_the_host(tmp_path, code, init)["dx"] - ref)) <= 4e-6 * np.max(np.abs(ref))


def _same_numbers(got, want, tol):
    """The same infinities and NaNs in the same places, and the rest within `tol` of the largest."""
    got = got.astype(np.float64)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    assert 0 < finite.sum() < want.size and np.max(np.abs(got[finite] - want[finite])) <= tol * np.max(np.abs(want[finite]))


def non_finite(nodes, seed):
    """Values for the nodes, an infinity or a NaN in some of the weights and gradients."""
    rng = np.random.default_rng(seed)
    init = {}
    for n in nodes:
        v = rng.standard_normal(n.dims).astype(np.float32)
        if n.ident != "dx":
            for x in (np.inf, -np.inf, np.nan):
                v.flat[rng.integers(v.size, size=2)] = x
        init[n.ident] = W.as_prec(v, n.prec)
    with np.errstate(invalid="ignore"):
        return init, {n.ident: W.to_float(init[n.ident], n.prec).astype(np.float64) for n in nodes}


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm compiler")
@pytest.mark.parametrize("prec", ["single", "bfloat16"])
@pytest.mark.parametrize("taps,stride,ic", [((3, 3), (1, 1), 33), ((3, 2), (2, 1), 40), ((5, 3), (2, 2), 5)])
@pytest.mark.parametrize("zeroed", [True, False])
def test_a_weight_counts_only_where_its_tap_reaches(taps, stride, ic, prec, zeroed, tmp_path):
    # 0 x infinity is NaN: a gathered position outside of a tap's reach has no such term
    r, nodes, want = input_gradient(taps, stride, prec, not zeroed, ic=ic, oc=8, zeroed=zeroed)
    init, values = non_finite(nodes, ic)
    with np.errstate(invalid="ignore"):
        ref = want(values)
    _same_numbers(_on_the_host(tmp_path, B.compile(r, "min_mfma_flops=1"), init)["dx"], ref, 4e-6)


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm compiler")
@pytest.mark.parametrize("prec", ["single", "bfloat16"])
@pytest.mark.parametrize("value,again", [(2.0 ** -149, False), (2.0 ** -111, False), (2.0 ** 70, False), (2.0 ** 105, True), (np.inf, True)])
def test_small_values_are_multiplied_once(value, again, prec, tmp_path):
    # an fp32 gradient of y of 288 products per cell, multiplied in bf16 parts: what soft-max tails hold costs no second pass
    r, (w, dy, dx), want = input_gradient((3, 3), (1, 1), prec, False, b=1, oh=4, ow=4)
    dy.prec = "single"
    rng = np.random.default_rng(8)
    init = {n.ident: W.as_prec(rng.standard_normal(n.dims).astype(np.float32), n.prec) for n in (w, dy, dx)}
    init["dy"].flat[::7] = value
    code = B.compile(r, "min_mfma_flops=1")
    assert ", true, 2, true>(d_" in code.source()
    out = _on_the_host(tmp_path, code, init)
    assert (out["f32_products"] > 0) == again
    with np.errstate(invalid="ignore"):
        ref = want({n.ident: W.to_float(init[n.ident], n.prec).astype(np.float64) for n in (w, dy, dx)})
    got, fine = out["dx"].astype(np.float64), np.isfinite(ref) & (np.abs(ref) < 2.0 ** 127)
    assert np.max(np.abs(got[fine] - ref[fine]), initial=0) <= 4e-6 * np.max(np.abs(ref[fine]), initial=0)   # (as above)
