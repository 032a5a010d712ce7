"""The C ABI library and its host-side logic (no GPU calls).

* every entry point declared in include/xyce_amd.h is exported;
* the host setup (node order, CSR pattern, stamp slots, state offsets) is
  bit-identical to the CPU oracle's for rings, inverter chains with internal
  drain/source nodes, power-grid meshes and gate DAGs;
* a hand-enumerated 3-stage ring pins both against the reference's stamp
  rules (jacStamp with RD=RS=0 merged, Vsrc branch row, ground dropped);
* the symbolic LU: valid permutations, zero-free diagonal, fill that equals
  a brute-force boolean elimination; a malformed pattern is rejected;
* a malformed circuit description (model, device or waveform index out of
  range, a device listed twice, a wrong count) is rejected with XG_E_SETUP;
* the patterns are one strongly connected block apart from each voltage
  source's two 1x1 blocks, so the block split of KLU's BTF would not change
  the ordering.
"""
import os
import re

import numpy as np
import pytest

import xyce_amd as X
from oracle.pyoracle import Oracle
from xyce_amd import circuits as C

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    hdr = open(os.path.join(ROOT, "include", "xyce_amd.h")).read()
    declared = set(re.findall(r"^int (xg_\w+)\(", hdr, flags=re.M))
    assert declared, "no declarations found"
    L = X.lib()
    missing = [s for s in sorted(declared) if not hasattr(L, s)]
    assert not missing, missing
    assert declared == set(X.EXPORTS)


def _same_pattern(c):
    hp = X.host_pattern(c)
    op = Oracle(c).pattern()
    for k in ("rowptr", "colind", "node_gid", "mos_lid", "mos_fslot", "mos_qslot", "mos_stasto"):
        assert np.array_equal(hp[k], op[k]), k
    return hp


@pytest.mark.parametrize("stages", [3, 5, 11, 53, 201])
def test_ring_pattern_matches_oracle(stages):
    _same_pattern(C.ring(stages, seed=stages, mc_seed=stages))


def test_internal_drain_source_nodes():
    c = C.inverter_chain(3, RD=25.0, RS=40.0, TOX=2e-8)
    hp = _same_pattern(c)
    # each MOSFET gains d' and s' unknowns: 6 MOSFETs x 2 + nodes + 2 branches
    assert hp["n"] == 6 * 2 + (c.n_nodes - 1) + 2
    assert np.all(hp["mos_lid"][:, 4] != hp["mos_lid"][:, 0])


def test_power_grid_and_dag_patterns_match_oracle():
    _same_pattern(C.power_grid(8, 8, seed=2, pad_pitch=4, n_sinks=5, tstop=1e-9))
    _same_pattern(C.gate_dag(60, seed=4))


def test_three_stage_ring_hand_enumerated():
    """Rows by the reference's stamp rules, independent of node numbering:
    out_k: {out_k-1, out_k, out_k+1, vdd};  vdd: {vdd, all outs, branch};
    branch: {vdd}."""
    c = C.ring(3, seed=1)
    hp = X.host_pattern(c)
    gid = hp["node_gid"]
    vdd = gid[1]
    outs = [gid[2 + k] for k in range(3)]
    bra = ({*range(hp["n"])} - {vdd, *outs}).pop()
    rows = {r: set(hp["colind"][hp["rowptr"][r]:hp["rowptr"][r + 1]]) for r in range(hp["n"])}
    for k in range(3):
        assert rows[outs[k]] == {outs[k - 1], outs[k], outs[(k + 1) % 3], vdd}
    assert rows[vdd] == {vdd, *outs, bra}
    assert rows[bra] == {vdd}
    assert hp["nnz"] == 5 * 3 + 3
    # NMOS of stage 1: drain out_1, gate out_3, source/bulk ground (dummy slot -1)
    lid = hp["mos_lid"][0]
    assert lid[0] == outs[0] and lid[1] == outs[2] and lid[2] == hp["n"] and lid[3] == hp["n"]
    fs = hp["mos_fslot"][0]
    rp, ci = hp["rowptr"], hp["colind"]
    slot = lambda r, col: rp[r] + int(np.where(ci[rp[r]:rp[r + 1]] == col)[0][0])
    # f_DrainPrimeEquGateNodePtr (index 8) -> (out_1, out_3); source rows -> ground
    assert fs[8] == slot(outs[0], outs[2])
    assert fs[10] == slot(outs[0], outs[0])
    assert fs[12] == -1 and fs[16] == -1


def _dense_of(n, rp, ci, vals=None):
    A = np.zeros((n, n))
    for r in range(n):
        for k in range(rp[r], rp[r + 1]):
            A[r, ci[k]] = 1.0 if vals is None else vals[k]
    return A


@pytest.mark.parametrize("maker", [lambda: C.ring(7, seed=1), lambda: C.ring(41, seed=2),
                                   lambda: C.power_grid(6, 6, seed=2, pad_pitch=3, n_sinks=3),
                                   lambda: C.gate_dag(40, seed=1)])
def test_symbolic_lu(maker):
    c = maker()
    hp = X.host_pattern(c)
    n = hp["n"]
    s = X.host_lu_analyse(n, hp["rowptr"], hp["colind"])
    pr, pc = s["perm_row"], s["perm_col"]
    assert sorted(pr) == list(range(n)) and sorted(pc) == list(range(n))
    A = _dense_of(n, hp["rowptr"], hp["colind"]) != 0
    B = A[np.ix_(pr, pc)]
    assert np.all(np.diag(B)), "transversal left a structural zero on the diagonal"
    # brute-force fill of the symmetric pattern of B
    F = B | B.T
    for k in range(n):
        rows = np.where(F[k + 1:, k])[0] + k + 1
        cols = np.where(F[k, k + 1:])[0] + k + 1
        F[np.ix_(rows, cols)] = True
    P = np.zeros((n, n), bool)
    lrp, lci = s["lu_rowptr"], s["lu_colind"]
    for i in range(n):
        P[i, lci[lrp[i]:lrp[i + 1]]] = True
    assert np.array_equal(P, F)
    assert s["nnz_lu"] == int(F.sum())


def test_value_steered_transversal_avoids_tiny_diagonal():
    """With values, a diagonal far below its column maximum is not used as a
    pivot (the ring at its DC point: gmin-sized diagonals, gm off-diagonals)."""
    n = 4
    # cyclic matrix with tiny diagonal
    rp = np.array([0, 2, 4, 6, 8], np.int32)
    ci = np.array([0, 3, 0, 1, 1, 2, 2, 3], np.int32)
    vals = np.array([1e-12, 1e-4, 1e-4, 1e-12, 1e-4, 1e-12, 1e-4, 1e-12])
    s = X.host_lu_analyse(n, rp, ci, values=vals)
    A = _dense_of(n, rp, ci, vals)
    B = A[np.ix_(s["perm_row"], s["perm_col"])]
    assert np.all(np.abs(np.diag(B)) >= 1e-4)


@pytest.mark.parametrize("case", ["col_high", "col_negative", "rowptr_decreasing", "rowptr_start"])
def test_malformed_pattern_is_rejected(case):
    """The symbolic analysis (what xg_lu_symbolic runs before any device
    work) rejects a malformed CSR pattern with XG_E_ARG instead of reading
    out of bounds."""
    rp = np.array([0, 2, 4, 6], np.int32)
    ci = np.array([0, 1, 0, 1, 1, 2], np.int32)
    if case == "col_high":
        ci[3] = 3
    elif case == "col_negative":
        ci[0] = -1
    elif case == "rowptr_decreasing":
        rp[2] = 1
    else:
        rp = rp + 1
    with pytest.raises(X.XgError, match="bad argument"):
        X.host_lu_analyse(3, rp, ci)
    X.host_lu_analyse(3, np.array([0, 2, 4, 6], np.int32), np.array([0, 1, 0, 1, 1, 2], np.int32))


@pytest.mark.parametrize("name", ["rings", "grids", "gates", "star", "clique", "path", "diagonal"])
def test_multifrontal_plan_covers_every_column(name):
    """The plan of systems around the dissection's leaf size (64) and of extreme
    shapes: built, every front square and within the system, at least the
    factor entries a dense diagonal needs."""
    def csr(M):
        rp = np.concatenate([[0], np.cumsum(M.sum(1))]).astype(np.int32)
        return M.shape[0], rp, np.nonzero(M)[1].astype(np.int32)
    if name == "star":
        pats = []
        for n in (2, 65, 200):
            M = np.eye(n, dtype=int); M[0] = 1; M[:, 0] = 1
            pats.append(csr(M))
    elif name == "clique":
        pats = [csr(np.ones((n, n), int)) for n in (1, 64, 65, 90)]
    elif name == "path":
        pats = [csr(np.eye(n, dtype=int) + np.eye(n, k=1, dtype=int) + np.eye(n, k=-1, dtype=int)) for n in (64, 65, 66, 300, 2000)]
    elif name == "diagonal":
        pats = [(n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)) for n in (1, 64, 65, 200_000)]
    else:
        cs = {"rings": [C.ring(s) for s in range(3, 140, 2)],
              "grids": [C.power_grid(a, b, pad_pitch=4, n_sinks=4) for a, b in ((1, 70), (2, 33), (8, 8), (9, 8), (33, 40))],
              "gates": [C.gate_dag(k, seed=k) for k in (20, 40, 45, 300, 1100)]}[name]
        hp = [X.host_pattern(c) for c in cs]
        pats = [(h["n"], h["rowptr"], h["colind"]) for h in hp]
    for n, rp, ci in pats:
        p = X.host_mf_plan(n, rp, ci)
        assert 1 <= p["supernodes"] <= n and 1 <= p["levels"] <= p["supernodes"] and 1 <= p["max_front"] <= n
        assert n <= p["nnz_lu"] <= p["front_elements"] and p["front_elements"] <= p["supernodes"] * p["max_front"] ** 2


@pytest.mark.parametrize("name", ["ring", "grid", "gates"])
def test_patterns_are_one_strongly_connected_block(name):
    import scipy.sparse as sp
    from scipy.sparse.csgraph import connected_components, maximum_bipartite_matching
    c = {"ring": lambda: C.ring(101),
         "grid": lambda: C.power_grid(40, 40, seed=7, pad_pitch=16, n_sinks=48),
         "gates": lambda: C.gate_dag(2000, seed=4)}[name]()
    p = X.host_pattern(c)
    n = p["n"]
    A = sp.csr_matrix((np.ones(len(p["colind"])), p["colind"], p["rowptr"]), shape=(n, n))
    match = maximum_bipartite_matching(A, perm_type="column")
    assert (match >= 0).all()
    k, lab = connected_components(A[:, match], directed=True, connection="strong")
    sizes = np.bincount(lab)
    n_vsrc = len(c.vsrc)
    assert k == 1 + 2 * n_vsrc and sizes.max() == n - 2 * n_vsrc


@pytest.mark.parametrize("corrupt", ["model_index", "device_twice", "device_index", "wave_index", "pulse_params",
                                     "n_dev", "node_id"])
def test_malformed_description_is_rejected(corrupt):
    """A description with an inconsistent count or index is rejected with
    XG_E_SETUP before anything is indexed with it."""
    import ctypes
    c = C.inverter_chain(2)
    d, a = X.make_desc(c)
    sizes = np.zeros(6, np.int32)
    call = lambda: X.lib().xg_host_pattern(ctypes.byref(d), sizes.ctypes.data_as(ctypes.c_void_p), None, None,
                                           None, None, None, None, None)
    assert call() == 0
    if corrupt == "model_index":
        a["mos_model"][1] = 7
    elif corrupt == "device_twice":
        a["dev_idx"][1] = a["dev_idx"][0]
        a["dev_type"][1] = a["dev_type"][0]
    elif corrupt == "device_index":
        a["dev_idx"][0] = 1000
    elif corrupt == "wave_index":
        a["vsrc_wave"][0] = 5
    elif corrupt == "pulse_params":
        k = int(np.nonzero(a["wave_type"] == C.W_PULSE)[0][0])
        d.n_wave = k + 1
        a["wave_off"][k + 1] = a["wave_off"][k] + 5
    elif corrupt == "n_dev":
        d.n_dev = d.n_dev - 1
    elif corrupt == "node_id":
        a["mos_nodes"][0] = d.n_nodes + 3
    assert call() == -3


@pytest.mark.parametrize("tstop,tstep,hmax,rec", [(0.0, 1e-12, 1e-11, 0), (1e-9, 0.0, 1e-11, 0),
                                                  (1e-9, 1e-12, -1.0, 0), (1e-9, 1e-12, 1e-11, -5),
                                                  (float("nan"), 1e-12, 1e-11, 0), (1e-9, float("inf"), 0.0, 0)])
def test_batch_create_rejects_bad_arguments(tstop, tstep, hmax, rec):
    """Out-of-range analysis arguments give XG_E_ARG before any device work
    (so also without a GPU); valid ones get past the check."""
    import ctypes
    d, keep = X.make_desc(C.ring(3, seed=1))
    h = ctypes.c_void_p()
    L = X.lib()
    dbl = ctypes.c_double
    assert L.xg_batch_create(1, ctypes.byref(d), dbl(tstop), dbl(tstep), dbl(hmax), rec, ctypes.byref(h)) == -1
    st = L.xg_batch_create(1, ctypes.byref(d), dbl(1e-9), dbl(1e-12), dbl(0.0), 0, ctypes.byref(h))
    assert st != -1
    if st == 0:
        L.xg_batch_destroy(h)


def test_multifrontal_analysis_without_threads():
    """Where no thread can be started (a stack limit larger than the address
    space) the plan is made by the calling thread, the same one."""
    import resource
    import subprocess
    import sys
    code = """
import sys, threading
sys.path.insert(0, %r)
import xyce_amd as X
from xyce_amd import circuits as C
try:
    threading.Thread(target=int).start()
    print("threads")
except RuntimeError:
    pass
h = X.host_pattern(C.power_grid(60, 60, seed=1, pad_pitch=16, n_sinks=16))
print(X.host_mf_plan(h["n"], h["rowptr"], h["colind"]))
""" % ROOT

    def limit():
        resource.setrlimit(resource.RLIMIT_STACK, (1 << 38, resource.RLIM_INFINITY))
        resource.setrlimit(resource.RLIMIT_AS, (1 << 36, 1 << 36))

    if resource.getrlimit(resource.RLIMIT_STACK)[1] not in (-1, resource.RLIM_INFINITY):
        pytest.skip("stack limit can't be raised")
    r = subprocess.run([sys.executable, "-c", code], preexec_fn=limit, capture_output=True, text=True,
                       env=dict(os.environ, OPENBLAS_NUM_THREADS="1", OMP_NUM_THREADS="1"))
    h = X.host_pattern(C.power_grid(60, 60, seed=1, pad_pitch=16, n_sinks=16))
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == str(X.host_mf_plan(h["n"], h["rowptr"], h["colind"]))
