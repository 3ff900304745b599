"""What the planner hands to the contraction tile for any shape, and what that tile reads; no GPU needed."""
import pytest

from ocannl_amd import backend as B
from ocannl_amd import llir as L


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
    # the tile's element offsets within one batch entry are ints: 2^20 * 1008 elements fit, 2^22 * 1008 do not
    assert "kernel_any<" in _matrix_kernels(_product(1008, 1008, 1 << 20, prec, *layout))[0]
    name, = _matrix_kernels(_product(1008, 1008, 1 << 22, prec, *layout))
    assert "kernel_any<" not in name


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
