"""Generated kernels at the edges of what a group of lanes is given: rows that are not a multiple of the lanes (kept in
registers, the last lanes with one position fewer), sums over short nested loops that all lanes share, the exchange
between 2 to 64 lanes, and whole routines in one workgroup whose tensors stay in LDS; against the CPU checker or one
thread per sum."""
import numpy as np
import pytest

from ocannl_amd import workloads as W
from parity import HipRun, OracleRun, rel_err

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
