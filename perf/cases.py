"""Performance cases of the framework: what a simulator built on it does all day.

Five kinds of work, each through the public entry points:

  loads   one device load of a Newton iteration (DeviceMgr): state update,
          vectors, matrices, residual and Jacobian; host arrays (the drop-in
          boundary) or device arrays (a caller that stays on the GPU)
  lu      one linear solve of a Newton iteration (DirectSolver): numeric
          refactor of new values and a solve, FP64 or FP32 with refinement
  tran    some time steps of one circuit on the resident engine (Transient)
  batch   Newton iterations of many independent circuits (Batch), then every
          instance's state read back
  mlp     the learned predictor's network: a forward pass (serving) or some
          training steps with the parameters read back

Circuits are the repository's own: ring oscillators, power-grid meshes and
INV/NAND2 gate arrays.  The structure of a case's circuit is fixed by its
sizes; device parameters, states and right-hand sides come from the seed.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import xyce_amd as X
from xyce_amd import circuits as C

VDD = C.VDD


def listed():
    return [
        # the smallest drop-in load: one 101-stage ring, host arrays, every call a few launches
        dict(name="loads_ring101", kind="loads", circuit="ring", size=101, form="host"),
        # a large gate array (about 300k MOSFETs) loaded by a caller that keeps its vectors on the GPU
        dict(name="loads_gates100k", kind="loads", circuit="gates", size=100_000, form="device"),
        # the smallest linear solve: KLU's place in a ring's Newton loop
        dict(name="lu_ring101", kind="lu", circuit="ring", size=101, form="host", fp32=False),
        # an ordinary, ragged power-grid mesh through host arrays
        dict(name="lu_grid131x97", kind="lu", circuit="grid", size=131, size2=97, form="host", fp32=False),
        # the full 512 x 512 mesh (262k unknowns), values and vectors on the GPU
        dict(name="lu_grid512", kind="lu", circuit="grid", size=512, size2=512, form="device", fp32=False),
        # a gate array's Jacobian with FP32 factors and FP64 refinement (150k unknowns)
        dict(name="lu_gates100k_fp32", kind="lu", circuit="gates", size=100_000, form="device", fp32=True),
        # time steps of a power grid on the resident engine (one Newton iteration a step)
        dict(name="tran_grid256", kind="tran", circuit="grid", size=256, size2=256, steps=4),
        # time steps of a switching gate array on the resident engine (several Newton iterations a step)
        dict(name="tran_gates2000", kind="tran", circuit="gates", size=2000, steps=8),
        # the Monte Carlo batch: 4096 rings of 11 to 201 stages
        dict(name="batch_mc4096", kind="batch", instances=4096, lo=11, hi=201, form="fused", block=256, launches=32),
        # one 101-stage ring alone on the batch engine
        dict(name="batch_ring101", kind="batch", instances=1, lo=101, hi=101, form="fused_lds", block=512, launches=8),
        # the predictor's network serving a batch of 4096 windows
        dict(name="mlp_serve4096", kind="mlp", rows=4096, width=512, hidden=3, train=0),
        # eight minibatches of the predictor's training at its default batch size
        dict(name="mlp_train2048", kind="mlp", rows=2048, width=512, hidden=3, train=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loads", "lu", "lu", "tran", "batch", "mlp"])
    if kind in ("loads", "lu"):
        c = dict(kind=kind, circuit=rng.choice(["ring", "grid", "gates"]), form=rng.choice(["host", "device"]))
        if c["circuit"] == "ring":
            c["size"] = 2 * _log_int(rng, 2, 250) + 1
        elif c["circuit"] == "grid":
            c["size"], c["size2"] = _log_int(rng, 8, 400), _log_int(rng, 8, 400)
        else:
            c["size"] = _log_int(rng, 40, 60_000)
        if kind == "lu":
            c["fp32"] = rng.random() < 0.3
        return c
    if kind == "tran":
        if rng.random() < 0.5:
            return dict(kind=kind, circuit="grid", size=_log_int(rng, 10, 250), size2=_log_int(rng, 10, 250),
                        steps=rng.randint(2, 4))
        return dict(kind=kind, circuit="gates", size=_log_int(rng, 50, 2000), steps=rng.randint(2, 8))
    if kind == "batch":
        lo = rng.randrange(5, 102, 2)
        return dict(kind=kind, instances=_log_int(rng, 1, 1024), lo=lo, hi=rng.randrange(lo, 202, 2),
                    form=rng.choice(["fused", "fused", "fused_lds", "split"]), block=rng.choice([128, 256]),
                    launches=rng.randint(2, 8))
    return dict(kind=kind, rows=64 * _log_int(rng, 1, 64), width=rng.choice([128, 256, 512]),
                hidden=rng.randint(1, 3), train=rng.choice([0, 0, 4, 8]))


# ----------------------------------------------------------------------
# circuits
# ----------------------------------------------------------------------
class _Arrays:
    """A circuit as the flat arrays that the library reads."""

    def __init__(self, a):
        self._a = a

    def arrays(self):
        return self._a


@functools.lru_cache(maxsize=4)
def _gate_arrays(size):
    return C.gate_dag(size, seed=4).arrays()


def _gates(size, seed):
    """A gate array with per-device threshold and transconductance spread and wire capacitances from the seed."""
    a = dict(_gate_arrays(size))
    rng = np.random.default_rng([seed, 1])
    inst = a["mos_inst"].reshape(-1, C.NIP).copy()
    pm = a["mos_model"] == 1
    inst[:, C.INST_PARAMS.index("VTO")] = np.where(pm, -0.7, 0.7) + 0.03 * rng.standard_normal(len(inst))
    inst[:, C.INST_PARAMS.index("KP")] = np.where(pm, 50e-6, 110e-6) * (1 + 0.05 * rng.standard_normal(len(inst)))
    a["mos_inst"] = inst.reshape(-1)
    a["cap_val"] = rng.uniform(0.5e-15, 5e-15, a["n_cap"])
    return _Arrays(a)


def _circuit(case, seed):
    if case["circuit"] == "ring":
        return C.ring(case["size"], seed=seed % 100_000 + 1, mc_seed=seed % 100_000 + 2)
    if case["circuit"] == "grid":
        nx, ny = case["size"], case["size2"]
        return C.power_grid(nx, ny, seed=seed % 100_000, pad_pitch=_pitch(nx, ny), n_sinks=_sinks(nx, ny))
    return _gates(case["size"], seed)


def _pitch(nx, ny):
    return max(4, min(64, min(nx, ny) // 2))


def _sinks(nx, ny):
    return max(4, nx * ny // 64)


def _grid_jacobian(case, seed, h=1e-12):
    """The transient Jacobian 0.5 G + C/h of a mesh with its pads' branch rows, as CSR arrays."""
    nx, ny = case["size"], case["size2"]
    rng = np.random.default_rng([seed, 2])
    ids = np.arange(nx * ny).reshape(ny, nx)
    gh = 0.5 / rng.uniform(0.05, 0.2, (ny, nx - 1))
    gv = 0.5 / rng.uniform(0.05, 0.2, (ny - 1, nx))
    dia = rng.uniform(10e-15, 100e-15, (ny, nx)) / h
    dia[:, :-1] += gh
    dia[:, 1:] += gh
    dia[:-1] += gv
    dia[1:] += gv
    p = _pitch(nx, ny)
    pads = ids[::p, ::p].reshape(-1)
    br = nx * ny + np.arange(len(pads))
    half = np.full(len(pads), 0.5)
    l, r, u, d = ids[:, :-1].reshape(-1), ids[:, 1:].reshape(-1), ids[:-1].reshape(-1), ids[1:].reshape(-1)
    row = np.concatenate([ids.reshape(-1), l, r, u, d, pads, br])
    col = np.concatenate([ids.reshape(-1), r, l, d, u, br, pads])
    gh, gv = gh.reshape(-1), gv.reshape(-1)
    val = np.concatenate([dia.reshape(-1), -gh, -gh, -gv, -gv, half, half])
    o = np.lexsort((col, row))
    n = nx * ny + len(pads)
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum(np.bincount(row, minlength=n))
    return n, rp, col[o].astype(np.int32), val[o]


def _state_of(d, rng, spread, h=2e-12):
    """Solver state of a transient Newton iteration, the point of the last one and what the devices kept from it."""
    d.set_solver_state(dcop=0, tran=1, newton_iter=1, order=2, h=h, time=0.4e-9, tstep=1e-12, tstop=2e-9)
    x0 = np.clip(0.5 * VDD + spread * rng.standard_normal(d.n), -0.2, VDD + 0.2)
    sta, sto, _ = d.updateState(x0, np.zeros(d.nsta), np.zeros(d.nsto))
    return x0, sta, sto


def _jacobian(case, seed):
    """(n, rowptr, colind, values) of a transient Jacobian."""
    if case["circuit"] == "grid":
        return _grid_jacobian(case, seed)
    d = X.DeviceMgr(_circuit(case, seed))
    _state_of(d, np.random.default_rng([seed, 3]), 0.05)
    v = d.loadDAEVectors()
    d.loadDAEMatrices()
    _, J = d.combine(v["Q"], v["F"] - v["B"])
    p = d.pattern()
    d.close()
    return d.n, p["rowptr"], p["colind"], J


def _solution(n, seed):
    return 0.05 * np.random.default_rng([seed, 4]).standard_normal(n)


# ----------------------------------------------------------------------
# prepare
# ----------------------------------------------------------------------
def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr() or None)


def prepare(case, seed):
    return dict(case=case, **{"loads": _prepare_loads, "lu": _prepare_lu, "tran": _prepare_tran,
                              "batch": _prepare_batch, "mlp": _prepare_mlp}[case["kind"]](case, seed))


def _prepare_loads(case, seed):
    rng = np.random.default_rng([seed, 5])
    d = X.DeviceMgr(_circuit(case, seed))
    x0, sta, sto = _state_of(d, rng, 0.5)
    v = d.loadDAEVectors()
    s = dict(d=d, x=x0 + 0.02 * rng.standard_normal(d.n), sta=sta, sto=sto, q0=v["Q"], q2=v["F"] - v["B"])
    if case["form"] == "device":
        for k in ("x", "sta", "sto", "q0", "q2"):
            s[k] = _gpu(s[k])
        s["sta_next"], s["sto_next"] = torch.zeros_like(s["sta"]), s["sto"].clone()
        s["out"] = torch.zeros(5 * d.n + 2 * d.nnz, dtype=torch.float64, device="cuda")
        s["rhs"] = torch.zeros(d.n, dtype=torch.float64, device="cuda")
        s["J"] = torch.zeros(d.nnz, dtype=torch.float64, device="cuda")
    return s


def _prepare_lu(case, seed):
    n, rp, ci, J = _jacobian(case, seed)
    # b = A x in extended precision, so that x is the solution to the last bits of b
    b = np.add.reduceat(J.astype(np.longdouble) * _solution(n, seed)[ci], rp[:-1]).astype(np.float64)
    s = X.DirectSolver(n, rp, ci)
    if case["fp32"]:
        s.set_precision(1)
    if case["form"] == "host":
        return dict(s=s, J=J, b=b)
    return dict(s=s, J=_gpu(J), b=_gpu(b), x=torch.zeros(n, dtype=torch.float64, device="cuda"))


def _prepare_tran(case, seed):
    if case["circuit"] == "grid":
        e = X.Transient(_circuit(case, seed), 2e-9, 1e-12, 1e-12)
        e.run(max_steps=1)          # the operating point and the first step
    else:
        e = X.Transient(_circuit(case, seed), 100e-9, 1e-12, 1e-11)
        e.set_uic()
        e.run(max_steps=16)         # the first edges of the power-up
    return dict(e=e)


def _prepare_batch(case, seed):
    stages = C.mc_stage_counts(case["instances"], lo=case["lo"], hi=case["hi"])
    at = 1000 + seed % 100_000
    b = X.Batch([C.ring(int(s), seed=at + i, mc_seed=at + i) for i, s in enumerate(stages)], 200e-9, 1e-12, 1e-11)
    if case["form"] == "split":
        b.config(block=case["block"], split_eval=1)
    else:
        b.config(block=case["block"], iters_per_launch=64, split_eval=2 if case["form"] == "fused_lds" else 0,
                 concurrent_groups=1)
    return dict(b=b, n=[int(s) + 2 for s in stages])


def _net_dims(case):
    w, k = case["width"], case["hidden"]
    return [(X.PRED_FEAT if l == 0 else w, w if l < k else X.PRED_WIN) for l in range(k + 1)]


def _net_params(case, seed):
    rng = np.random.default_rng([seed, 7])
    p = []
    for di, do in _net_dims(case):
        p += [rng.uniform(-1, 1, (do, di)) / math.sqrt(di), 0.02 * rng.standard_normal(do)]
    return [v.astype(np.float32) for v in p]


def _net_data(case, seed):
    """Features in the predictor's compressed units, targets in Newton weights, the last rows of each window unused."""
    g = torch.Generator().manual_seed(seed % (1 << 40))
    r = case["rows"]
    x = (2.0 * torch.randn(r, X.PRED_FEAT, generator=g)).to(torch.bfloat16)
    t = 0.5 * torch.randn(r, X.PRED_WIN, generator=g)
    used = torch.randint(13, X.PRED_WIN + 1, (r, 1), generator=g)
    m = (torch.arange(X.PRED_WIN)[None] < used).float()
    return x, t, m


def _prepare_mlp(case, seed):
    net = X.MLP(X.PRED_FEAT, case["width"], case["hidden"], X.PRED_WIN, max_rows=case["rows"])
    p = np.concatenate([v.reshape(-1) for v in _net_params(case, seed)])
    net.set_params(p)
    x, t, m = _net_data(case, seed)
    s = dict(net=net, x=x.cuda())
    if case["train"]:
        s.update(t=t.cuda(), m=m.cuda(), count=int(m.sum()))
    else:
        s["y"] = torch.zeros(case["rows"], X.PRED_WIN, device="cuda")
    return s


# ----------------------------------------------------------------------
# run
# ----------------------------------------------------------------------
def run(s):
    return {"loads": _run_loads, "lu": _run_lu, "tran": _run_tran, "batch": _run_batch,
            "mlp": _run_mlp}[s["case"]["kind"]](s)


def _ok(status):
    if status != 0:
        raise RuntimeError("status %d" % status)


def _run_loads(s):
    d = s["d"]
    if s["case"]["form"] == "host":
        sta, sto, limited = d.updateState(s["x"], s["sta"], s["sto"])
        v = d.loadDAEVectors()
        dF, dQ = d.loadDAEMatrices()
        rhs, J = d.combine(s["q0"], s["q2"])
        return dict(v, sta=sta, sto=sto, limited=limited, dFdx=dF, dQdx=dQ, rhs=rhs, J=J)
    L = X.lib()
    limited = ctypes.c_int(0)
    out = s["out"].zero_()      # the loader's zeroed vectors and matrices, which the devices add to
    n, nnz = d.n, d.nnz
    vec = [out[i * n:(i + 1) * n] for i in range(5)]
    mat = [out[5 * n + i * nnz:5 * n + (i + 1) * nnz] for i in range(2)]
    _ok(L.xg_update_state_dev(d.h, _ptr(s["x"]), _ptr(s["sta"]), _ptr(s["sto"]), _ptr(s["sta_next"]),
                              _ptr(s["sto_next"]), ctypes.byref(limited)))
    _ok(L.xg_load_vectors_dev(d.h, *[_ptr(v) for v in vec]))
    _ok(L.xg_load_matrices_dev(d.h, *[_ptr(v) for v in mat]))
    _ok(L.xg_combine_dev(d.h, _ptr(s["q0"]), _ptr(s["q2"]), _ptr(s["rhs"]), _ptr(s["J"])))
    return dict(F=vec[0], Q=vec[1], B=vec[2], FL=vec[3], QL=vec[4], dFdx=mat[0], dQdx=mat[1], sta=s["sta_next"],
                sto=s["sto_next"], limited=limited.value, rhs=s["rhs"], J=s["J"])


def _run_lu(s):
    if s["case"]["form"] == "host":
        status, x = s["s"].doSolve(s["J"], s["b"])
        _ok(status)
        return dict(x=x)
    L = X.lib()
    _ok(L.xg_lu_numeric_dev(s["s"].h, _ptr(s["J"])))
    _ok(L.xg_lu_solve_dev(s["s"].h, _ptr(s["b"]), _ptr(s["x"]), 0))
    return dict(x=s["x"])


def _run_tran(s):
    r = s["e"].run(max_steps=s["case"]["steps"])
    return dict(x=s["e"].solution(), t=r["t"], steps=r["steps"], rejects=r["rejects"], newton=r["newton_iters"],
                status=r["status"])


def _run_batch(s):
    b, case = s["b"], s["case"]
    b.advance(case["launches"] if case["form"] != "split" else 64 * case["launches"])
    state, x = zip(*(b.instance(i, n) for i, n in enumerate(s["n"])))
    return dict(x=np.concatenate(x), t=np.array([v["t"] for v in state]), h=np.array([v["h"] for v in state]),
                counts=np.array([[int(v[k]) for k in ("mode", "newton_iters", "steps", "rejects", "loads")]
                                 for v in state]))


def _run_mlp(s):
    net = s["net"]
    if not s["case"]["train"]:
        net.forward(s["x"], s["y"])
        return dict(y=s["y"])
    loss = []
    for _ in range(s["case"]["train"]):
        loss.append(net.loss_backward(s["x"], s["t"], s["m"], s["count"]))
        net.adam(1e-3)
    net.sync()
    # the loss is a sum over the network's FP32 outputs
    return dict(loss=np.array(loss, np.float32), params=net.params())


# ----------------------------------------------------------------------
# work and exact results
# ----------------------------------------------------------------------
@functools.lru_cache(maxsize=16)
def _sizes(circuit, size, size2):
    """(unknowns, CSR entries, MOSFETs, factor entries, flops of a factorisation) of a circuit."""
    case = dict(circuit=circuit, size=size, size2=size2)
    if circuit == "grid":
        n, rp, ci, _ = _grid_jacobian(case, 0)
        n_mos = 0
    else:
        p = X.host_pattern(_circuit(case, 0))
        n, rp, ci, n_mos = p["n"], p["rowptr"], p["colind"], len(p["mos_lid"])
    plan = X.host_mf_plan(n, rp, ci)
    return n, len(ci), n_mos, plan["nnz_lu"], plan["flops"]


#: floating-point operations of one level-1 MOSFET evaluation, about (square roots and exponentials counted as 20)
MOS_FLOPS = 400


def _loads_work(n, nnz, n_mos):
    # per MOSFET: three parameters, class and mask (36 B), six unknown numbers (24 B), the store at t_n and at the last
    # iterate and the state at t_n read (160 B), the next store and state written (112 B); x and two histories read,
    # five vectors and the residual written; the linear part read, dF/dx, dQ/dx and the Jacobian written
    return n_mos * (36 + 24 + 160 + 112) + n * 8 * (3 + 6) + nnz * 8 * (2 + 3), n_mos * MOS_FLOPS + 14 * n + 7 * nnz


def _lu_work(n, nnz, nlu, flops, width):
    # the values read, the factors written once and read once by the solve, b read and x written
    return nnz * 8 + nlu * 2 * width + n * 16, flops + 2 * nlu


def work(case):
    kind = case["kind"]
    if kind in ("loads", "lu", "tran"):
        n, nnz, n_mos, nlu, flops = _sizes(case["circuit"], case["size"], case.get("size2", 0))
        lb, lf = _loads_work(n, nnz, n_mos)
        if kind == "loads":
            return {"bytes": lb, "flops": lf}
        ub, uf = _lu_work(n, nnz, nlu, flops, 4 if case.get("fp32") else 8)
        if kind == "lu":
            return {"bytes": ub, "flops": uf}
        # one Newton iteration a step for a linear grid, about three for switching gates
        k = case["steps"] * (3 if n_mos else 1)
        return {"bytes": k * (lb + ub), "flops": k * (lf + uf)}
    if kind == "batch":
        # means over the stage counts: 2 MOSFETs, 1 unknown and 5 entries a stage, 9 factor entries, 36 flops of LU
        m = case["instances"] * 0.5 * (case["lo"] + case["hi"]) * 64 * case["launches"]
        return {"bytes": m * (2 * 308 + 56 + 5 * 16), "flops": m * (2 * MOS_FLOPS + 36 + 4 * 9 + 60)}
    p = sum(di * do + do for di, do in _net_dims(case))
    r = case["rows"]
    io = r * X.PRED_FEAT * 2 + r * X.PRED_WIN * 4
    if not case["train"]:
        return {"bytes": io + 2 * p, "flops": 2 * r * p}
    # forward and both backward products (the first layer's input needs no gradient); parameters and moments updated
    first = X.PRED_FEAT * case["width"]
    one = {"bytes": io + r * X.PRED_WIN * 4 + p * (2 + 4 + 6 * 4), "flops": 2 * r * (3 * p - first)}
    return {k: case["train"] * v for k, v in one.items()}


def exact(case, seed):
    """64-bit results: the solution that a linear system was made from, and the network in double precision.  The other
    outputs (device models, trajectories) have no value that plain array arithmetic gives."""
    if case["kind"] == "lu":
        if case["circuit"] == "grid":
            nx, ny = case["size"], case["size2"]
            p = _pitch(nx, ny)
            n = nx * ny + len(range(0, ny, p)) * len(range(0, nx, p))
        elif case["circuit"] == "ring":
            n = case["size"] + 2
        else:
            # nodes without ground, and a branch current per voltage source
            a = _gate_arrays(case["size"])
            n = a["n_nodes"] - 1 + a["n_vsrc"]
        return dict(x=_solution(n, seed))
    if case["kind"] != "mlp":
        return None
    x, t, m = _net_data(case, seed)
    x, t, m = x.double(), t.double(), m.double()
    p = [torch.from_numpy(v).double() for v in _net_params(case, seed)]

    def forward(weights):
        v = x
        for l in range(case["hidden"] + 1):
            v = v @ weights[2 * l].T + weights[2 * l + 1]
            if l < case["hidden"]:
                v = torch.nn.functional.gelu(v)
        return v

    if not case["train"]:
        # the network's weights are BF16 by definition
        return dict(y=forward([w.to(torch.bfloat16).double() if w.ndim == 2 else w for w in p]).numpy())
    if case["rows"] * case["train"] * sum(w.numel() for w in p) > 3e10:
        return None     # too long for a CPU
    m1, m2 = [torch.zeros_like(w) for w in p], [torch.zeros_like(w) for w in p]
    loss, b1, b2, count = [], 0.9, 0.999, float(m.sum())
    for k in range(1, case["train"] + 1):
        for w in p:
            w.requires_grad_(True)
        e = (((forward(p) - t) * m) ** 2).sum() / count
        g = torch.autograd.grad(e, p)
        loss.append(float(e.detach()))
        p = [w.detach() for w in p]
        for i in range(len(p)):
            m1[i] = b1 * m1[i] + (1 - b1) * g[i]
            m2[i] = b2 * m2[i] + (1 - b2) * g[i] ** 2
            p[i] = p[i] - 1e-3 * (m1[i] / (1 - b1 ** k)) / ((m2[i] / (1 - b2 ** k)).sqrt() + 1e-8)
    return dict(loss=np.array(loss), params=torch.cat([w.reshape(-1) for w in p]).numpy())
