"""Generated kernels at the edges of what a group of lanes is given: rows that are not a multiple of the lanes (kept in
registers, the last lanes with one position fewer), sums over short nested loops that all lanes share, the exchange
between 2 to 64 lanes, and whole routines in one workgroup whose tensors stay in LDS; against the CPU checker, one
thread per sum, or sums in float64."""
import numpy as np
import pytest
import torch  # noqa: F401  (its copy of the HIP runtime has to be loaded first)

from ocannl_amd import llir as L
from ocannl_amd import workloads as W
from parity import HipRun, OracleRun, rel_err, tensor_err
from test_gpu_models import _err, _widened_init

pytestmark = pytest.mark.gpu


def _agrees(w, statics, steps, names, tol=2e-4):
    ref, hip = OracleRun(w.routine, w.init), HipRun(w.routine, w.init)
    for s in range(steps):
        ref.step(statics(s)); hip.step(statics(s))
    for name in names:
        n = w.nodes[name]
        err = rel_err(hip.get(n), np.asarray(ref.get(n)).reshape(n.dims), n.prec)
        assert err <= tol, (name, err)
    hip.close()


@pytest.mark.parametrize("batch,hidden", [(1, 1), (3, 5), (20, 17), (61, 10), (33, 33), (9, 65), (128, 10)])
def test_one_workgroup(batch, hidden):
    w = W.moons_mlp(batch=batch, hidden=hidden)
    sym, nb = w.statics["batch_n"].sym, w.statics["batch_n"].range
    _agrees(w, lambda s: {sym: s % nb}, 3, ("loss", "w1", "b1", "w2", "b2", "w3", "mom_w2"))


@pytest.mark.parametrize("q,k,d", [(5, 17, 8), (7, 63, 9), (3, 65, 16), (9, 99, 7), (2, 1003, 8), (3, 1025, 5), (2, 1280, 4)])
def test_row_lengths(q, k, d):
    w = W.attention(b=1, h=2, q=q, k=k, d=d, prec="single", grad_prec="single")
    _agrees(w, lambda s: None, 1, ("out", "dq", "dk", "dv"))


@pytest.mark.parametrize("opts", ["serial=0", None])
@pytest.mark.parametrize("q,k,d", [(7, 63, 9), (9, 99, 7), (197, 197, 16), (2, 1003, 8), (64, 1025, 5)])
def test_row_lengths_in_bf16(q, k, d, opts):
    # Against the oracle in fp32 on the same values: 2e-2 in the Frobenius norm as every bf16 routine, and no element
    # further off than 2^-5 of the tensor's largest -- scores, exponentials, weights and their gradients carry up to
    # sixteen roundings of 2^-9, and a gradient is a sum of few terms that cancel, so its own row sets no scale.
    w, wr = (W.attention(b=1, h=2, q=q, k=k, d=d, prec=p, grad_prec="single") for p in ("bfloat16", "single"))
    hip, ref = HipRun(w.routine, w.init, opts), OracleRun(wr.routine, _widened_init(w, wr))
    hip.step(); ref.step()
    if opts:   # (not in the one workgroup of a tiny routine: rows in registers, the last lanes one position short)
        assert f"> {k - 1}) continue;" in hip.code.source()
    for name, p in (("out", "bfloat16"), ("dq", "single"), ("dk", "single"), ("dv", "single")):
        n = wr.nodes[name]
        got, want = W.to_float(hip.get(w.nodes[name]), p), np.asarray(ref.get(n)).reshape(n.dims)
        assert _err(got, want, "bfloat16") <= 2e-2 and tensor_err(got, want, "double") <= 2.0 ** -5, name
    hip.close()


@pytest.mark.parametrize("batch,vocab", [(2, 3), (5, 27), (33, 9), (64, 70)])   # losses summed over batch x vocab
def test_nested_sums(batch, vocab):
    """Against one thread per sum (the CPU checker's compiler breaks the guarded gather on hosts with AVX-512)."""
    w = W.char_mlp(batch=batch, vocab=vocab, hidden=40, embed=5)
    ref, hip = HipRun(w.routine, w.init, "coop=0;rows=0;serial=0;parallel=0"), HipRun(w.routine, w.init)
    for s in range(2):
        st = {v.sym: s for v in w.statics.values()}
        ref.step(st); hip.step(st)
    for name in ("loss", "c", "w1", "b2", "m_w1", "v_w2"):
        err = rel_err(hip.get(w.nodes[name]), ref.get(w.nodes[name]), "single")
        assert err <= 2e-4, (name, err)
    ref.close(); hip.close()


@pytest.mark.parametrize("inlined", [False, True])
@pytest.mark.parametrize("points,n,m", [(1, 33, 7), (3, 1000, 40), (5, 65, 63), (16, 409, 5), (17, 300, 2), (2, 64, 64)])
def test_nested_sums_in_float64(points, n, m, inlined):
    # out[p] = sum over i and j of a[p, i] * b[i, j]: lanes outnumber the inner loop, up to a whole workgroup a sum
    L.reset_symbols(0)
    a, b, out = L.Node(1, "a", "single", (points, n)), L.Node(2, "b", "single", (n, m)), L.Node(3, "out", "single", (points,))
    p, i, j = (L.fresh_symbol() for _ in range(3))
    at = (L.It(p),)
    term = lambda acc: L.Ternop("fma", L.Get(a, (L.It(p), L.It(i))), L.Get(b, (L.It(i), L.It(j))), acc)
    loops = lambda body: L.For(i, 0, n - 1, [L.For(j, 0, m - 1, [body])])
    if inlined:
        v = L.Scope(L.Node(4, "v", "single", (points,), mode="virtual"), L.fresh_symbol())
        body = [L.For(p, 0, points - 1, [L.Set(out, at, L.LocalScope(v, [L.SetLocal(v, L.Const(0.0)), loops(L.SetLocal(v, term(L.GetLocal(v))))]))])]
    else:
        body = [L.ZeroOut(out), L.For(p, 0, points - 1, [loops(L.Set(out, at, term(L.Get(out, at))))])]
    rng = np.random.default_rng(n)
    init = {x.id: rng.standard_normal(x.dims).astype(np.float32) for x in (a, b)}
    hip = HipRun(L.Routine("nested", body), init, "mfma=0;serial=0")
    hip.step()
    terms = init[1].astype(np.float64)[:, :, None] * init[2].astype(np.float64)[None]
    # at least 64 lanes: a term goes through at most n * m / 64 roundings in its lane and 8 between lanes, each below 2^-24
    # of the sum of absolute values
    bound = np.abs(terms).sum(axis=(1, 2)) * (n * m / 64 + 9) * 2.0 ** -24
    assert np.all(np.abs(hip.get(out) - terms.sum(axis=(1, 2))) <= bound)
    hip.close()
