"""The framework's performance cases: what its users have it do, through its
public entry points (amat_amd: Maps, aMatFree, MultiRHS, Server).

listed() names the fixed cases, draw(rng) makes further ones over the same
ranges, prepare(case, seed) builds what a program holds before the call (the
finalized operator, its vectors on the GPU), run(state) makes one call,
work(case) counts the bytes and flops of that call that no implementation can
do without, and exact(case, seed) gives its outputs in 64 bits in plain numpy.

Kinds of case ("what"):
  matvec    one operator application on device vectors with element matrices
            given to the operator: K_e = s_e K_ref ("scaled": hex8 Poisson and
            hex20 elasticity on congruent meshes) or one matrix per element
            ("distinct": jittered tet10 Poisson with a coefficient per element,
            hex20 elasticity of mixed element shapes), stored in FP64, FP32 or BF16.
  method2   the same product recomputed from the node coordinates.
  solve     a whole conjugate-gradient solve to 1e-10: FP64, or FP32 / BF16
            element matrices with FP64 residual replacements.
  multirhs  one launch of several right-hand sides over two meshes.
  serve     a batch of CG requests of mixed meshes through the solve server.
"""
from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

from amat_amd import BCOP, ELEM, PREC, SCATTER, Maps, MultiRHS, aMatFree, fem, mesh, problems
from amat_amd.amat import IR_RELIABLE
from amat_amd.serve import Server

DOFS = {"hex8": 8, "hex20": 60, "tet10": 10}
BCS = {"none": BCOP.NONE, "identity": BCOP.IDENTITY, "penalty": BCOP.PENALTY_DIAG}
PRECS = {"fp64": PREC.FP64, "fp32": PREC.FP32, "bf16": PREC.BF16}
PENALTY = 1e8
SHAPES = 16  # element shapes of the mixed hex20 meshes


def listed() -> list[dict]:
    return [
        # the smallest call: a Poisson matvec whose two launches take longer than its data; what a
        # CG on a small mesh repeats
        _matvec("poisson_hex8_32", "hex8", 32, bc="identity"),
        # the product the framework is bought for: hex20 elasticity at real size
        _matvec("elasticity_hex20_64", "hex20", 64, bc="penalty"),
        # elasticity with a matrix per element (mixed shapes), as an unstructured mesh gives them
        _matvec("elasticity_hex20_distinct_24", "hex20", 24, matrices="distinct", bc="identity"),
        # Poisson on a jittered tet10 mesh, every matrix its own; an odd and a round size, the FP64
        # product and the BF16 one of the mixed-precision solvers
        _matvec("poisson_tet10_48", "tet10", 48, matrices="distinct", bc="identity"),
        _matvec("poisson_tet10_33_bf16", "tet10", 33, matrices="distinct", bc="identity", prec="bf16"),
        # matrix-free products from coordinates: elasticity with the full 27-point rule, Poisson on tets
        {"name": "method2_hex20_48_ngt3", "what": "method2", "mesh": "hex20", "n": 48, "ngt": 3, "bc": "identity",
         "prec": "fp64"},
        {"name": "method2_tet10_41", "what": "method2", "mesh": "tet10", "n": 41, "ngt": 2, "bc": "identity",
         "prec": "fp64"},
        # whole solves: plain FP64 CG of a Poisson problem, mixed precision on elasticity
        {"name": "solve_hex8_48_fp64", "what": "solve", "mesh": "hex8", "n": 48, "method": "fp64"},
        {"name": "solve_hex20_15_fp32r", "what": "solve", "mesh": "hex20", "n": 15, "method": "fp32r"},
        # blocks of right-hand sides: many in FP32 summed in a fixed order, few in BF16 with atomics
        {"name": "multirhs_fp32_128", "what": "multirhs", "n": 32, "hx": 40, "hy": 20, "hz": 10, "nrhs": 128,
         "prec": "fp32", "scatter": "fixed"},
        {"name": "multirhs_bf16_24", "what": "multirhs", "n": 31, "hx": 80, "hy": 40, "hz": 20, "nrhs": 24,
         "prec": "bf16", "scatter": "atomic"},
        # a batch of requests as the solve server takes them
        {"name": "serve_mix_12", "what": "serve", "count": 12, "pick": 7, "method": "fp64"},
    ]


def _matvec(name, kind, n, ny=0, nz=0, matrices="scaled", bc="none", prec="fp64", scatter="fixed") -> dict:
    """ny, nz: elements along y and z (0: n)."""
    return {"name": name, "what": "matvec", "mesh": kind, "n": n, "ny": ny, "nz": nz, "matrices": matrices, "bc": bc,
            "prec": prec, "scatter": scatter}


def draw(rng: random.Random) -> dict:
    def size(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    kind = rng.choice(["matvec", "matvec", "matvec", "method2", "solve", "multirhs", "serve"])
    if kind == "matvec":
        which = rng.choice(["hex8", "hex20", "hex20", "hex20distinct", "tet10"])
        m = which[:5]
        n = size(*{"hex8": (12, 96), "hex20": (5, 56), "hex20distinct": (4, 24), "tet10": (6, 44)}[which])
        ny, nz = (size(max(2, n // 2), n), size(max(2, n // 2), n)) if m != "tet10" else (0, 0)
        c = _matvec("", m, n, ny, nz, "scaled" if which in ("hex8", "hex20") else "distinct",
                    rng.choice(["none", "identity", "identity", "penalty"]), rng.choice(["fp64", "fp64", "fp32", "bf16"]),
                    rng.choice(["fixed", "fixed", "fixed", "atomic"]))
    elif kind == "method2":
        m = rng.choice(["hex8", "hex20", "hex20", "tet10"])
        n = size(*{"hex8": (12, 80), "hex20": (5, 44), "tet10": (6, 38)}[m])
        c = {"what": kind, "mesh": m, "n": n, "ngt": rng.choice([2, 3]) if m == "hex20" else 2,
             "bc": rng.choice(["none", "identity", "penalty"]), "prec": rng.choice(["fp64", "fp64", "fp32"])}
    elif kind == "solve":
        m = rng.choice(["hex8", "hex20", "tet10"])
        n = size(*{"hex8": (16, 64), "hex20": (5, 15), "tet10": (8, 24)}[m])
        c = {"what": kind, "mesh": m, "n": n,
             "method": rng.choice(["fp64", "fp32r"] + ([] if m == "hex20" else ["bf16r"]))}
    elif kind == "multirhs":
        nrhs = rng.choice([1, 3, 8, 17, 32, 50, 64, 100, 128])
        c = {"what": kind, "n": size(6, 31), "hx": size(8, 80), "hy": size(8, 40), "hz": size(4, 20), "nrhs": nrhs,
             "prec": rng.choice(["fp32", "bf16"]), "scatter": rng.choice(["fixed", "atomic"])}
    else:
        c = {"what": kind, "count": rng.randint(3, 11), "pick": rng.randint(1, 999),
             "method": rng.choice(["fp64", "fp32r"])}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ problems
@functools.lru_cache(maxsize=16)
def _problem(kind: str, n: int, ny: int, nz: int, ngt: int = 2) -> problems.Problem:
    """Mesh, maps and reference matrices; nothing here depends on a seed."""
    if kind == "hex8":
        return problems.poisson_hex8(n, ny or None, nz or None)
    if kind == "hex20":
        return problems.elasticity_hex20(n, ny or None, nz or None, ngt=max(ngt, 2), perturb=False)
    return problems.poisson_tet10(n, with_rhs=False)


@functools.lru_cache(maxsize=1)
def _hex20_shapes() -> np.ndarray:
    """Elasticity matrices of SHAPES distorted hexahedra."""
    m = mesh.hex20(1, 1, 1)
    x = m.coords[m.elem_nodes[0]]
    return np.stack([fem.ke_hex20_iso(x + mesh.uniform(31 + i, 3, 60, -0.04, 0.04).reshape(20, 3), 1.0, 0.3, 3)
                     for i in range(SHAPES)])


def _scales(case: dict, p: problems.Problem, seed: int) -> np.ndarray:
    """Stiffness per element: 1 for the hex8 Poisson problem, U[0.5, 2) otherwise."""
    if case["mesh"] == "hex8":
        return np.ones(p.n_elem)
    return mesh.uniform(seed, 2, p.n_elem, 0.5, 2.0)


def _matrices(case: dict, p: problems.Problem, seed: int) -> np.ndarray:
    s = _scales(case, p, seed)
    if case["mesh"] == "tet10":
        return p.K * s[:, None, None]
    which = (mesh.uniform(seed, 4, p.n_elem) * SHAPES).astype(np.int64)
    return _hex20_shapes()[which] * s[:, None, None]


def _operator(case: dict, p: problems.Problem, seed: int, precision: int = int(PREC.FP64)) -> aMatFree:
    op = aMatFree(p.build_maps(Maps))
    if case["what"] == "method2":
        op.set_matfree_type(2)
        f = p.free
        op.set_element_function(ELEM(f["kind"]), _coords(case, p, seed), _scales(case, p, seed), f.get("E", 1.0),
                                f.get("nu", 0.3), case["ngt"])
    elif case.get("matrices", "scaled" if p.K is None else "distinct") == "scaled":
        op.set_element_matrices_scaled(p.k_ref, _scales(case, p, seed))
    else:
        op.set_element_matrices(0, _matrices(case, p, seed))
    op.set_options(precision, SCATTER.ATOMIC if case.get("scatter") == "atomic" else SCATTER.DETERMINISTIC)
    bc = case.get("bc", "identity")
    op.set_bc_operator(BCS[bc])
    if bc == "penalty":
        op.set_penalty(PENALTY)
    op.finalize()
    return op


def _coords(case: dict, p: problems.Problem, seed: int) -> np.ndarray:
    """Node coordinates per element; on hexahedra every node moved by up to 2 % of the
    element size (the tet10 meshes are jittered already)."""
    h = 1.0 / case["n"] if case["mesh"] != "tet10" else 0.0
    x = p.mesh.coords + mesh.uniform(seed, 6, 3 * p.mesh.n_nodes, -0.02 * h, 0.02 * h).reshape(-1, 3)
    return np.ascontiguousarray(x[p.mesh.elem_nodes])


def _rhs(p: problems.Problem, seed: int) -> np.ndarray:
    b = mesh.uniform(seed, 5, p.n_dofs, -1.0, 1.0)
    b[p.constrained.astype(np.int64)] = 0.0
    return b


def _of(case: dict) -> problems.Problem:
    return _problem(case["mesh"], case["n"], case.get("ny", 0), case.get("nz", 0), case.get("ngt", 3))


def _multirhs(case: dict, seed: int):
    """[(problem, scales, U)] of the two meshes of a multi-RHS call."""
    out = []
    for i, (kind, dims) in enumerate((("hex20", (case["n"], 0, 0)), ("hex8", (case["hx"], case["hy"], case["hz"])))):
        p = _problem(kind, *dims, 3)
        U = mesh.uniform(seed, 10 + i, p.n_dofs * case["nrhs"], -1.0, 1.0).astype(np.float32)
        out.append((p, _scales({"mesh": kind}, p, seed + i), U.reshape(p.n_dofs, case["nrhs"])))
    return out


def _requests(case: dict) -> list[dict]:
    """The served mix: 60 % hex8, 30 % hex20, 10 % tet10, sizes of a small server."""
    r = random.Random(case["pick"])
    out = []
    for _ in range(case["count"]):
        x = r.random()
        kind, lo, hi = ("hex8", 16, 48) if x < 0.6 else ("hex20", 8, 14) if x < 0.9 else ("tet10", 12, 18)
        out.append({"what": "solve", "mesh": kind, "n": r.randint(lo, hi), "method": case["method"]})
    return out


# ------------------------------------------------------------------ the cases
def _method(name: str) -> tuple[int, int]:
    """(storage mask, solver method) of a solve."""
    if name == "fp64":
        return int(PREC.FP64), int(PREC.FP64)
    low = PRECS[name[:4]]
    return int(PREC.FP64 | low), int(low) | IR_RELIABLE


def prepare(case: dict, seed: int):
    st = {"what": case["what"]}
    if case["what"] in ("matvec", "method2"):
        p = _of(case)
        prec = PRECS[case["prec"]]
        stored = PREC.FP64 if case["what"] == "method2" else PREC.FP64 | prec
        st["op"], st["prec"] = _operator(case, p, seed, int(stored)), prec
        u = mesh.uniform(seed, 1, p.n_dofs, -1.0, 1.0)
        st["u"] = torch.from_numpy(u).cuda().to(torch.float64 if prec == PREC.FP64 else torch.float32)
        st["v"] = torch.empty_like(st["u"])
    elif case["what"] == "solve":
        p = _of(case)
        mask, st["method"] = _method(case["method"])
        st["op"] = _operator(case, p, seed, mask)
        st["b"] = torch.from_numpy(_rhs(p, seed)).cuda()
        st["x"] = torch.zeros_like(st["b"])
    elif case["what"] == "multirhs":
        parts = _multirhs(case, seed)
        ops = []
        for p, s, _ in parts:
            op = aMatFree(p.build_maps(Maps))
            op.set_element_matrices_scaled(p.k_ref, s)
            op.finalize()
            ops.append(op)
        st["nrhs"] = case["nrhs"]
        st["mr"] = MultiRHS(ops, PRECS[case["prec"]])
        st["mr"].set_scatter(SCATTER.ATOMIC if case["scatter"] == "atomic" else SCATTER.DETERMINISTIC)
        st["U"] = [torch.from_numpy(U).cuda() for _, _, U in parts]
        st["V"] = [torch.empty_like(U) for U in st["U"]]
        st["mr"].autotune(case["nrhs"], st["U"], st["V"], reps=3, stream=torch.cuda.current_stream())
    else:
        st["server"] = Server(max_jobs=32)
        st["jobs"] = []
        for i, r in enumerate(_requests(case)):
            p = _of(r)
            mask, method = _method(r["method"])
            st["jobs"].append((_operator(r, p, seed + i, mask), method, _rhs(p, seed + i)))
    return st


def run(st):
    s = torch.cuda.current_stream()
    if st["what"] in ("matvec", "method2"):
        if st["prec"] == PREC.FP64:
            st["op"].matmult_dev(st["v"], st["u"], s)
        else:
            st["op"].matmult_f32_dev(st["prec"], st["v"], st["u"], s)
        return st["v"]
    if st["what"] == "solve":
        if st["method"] == int(PREC.FP64):
            st["op"].cg(st["b"], st["x"], rtol=1e-10, stream=s)
        else:
            st["op"].ir_cg(st["method"], st["b"], st["x"], rtol=1e-10, inner_rtol=0.1, max_outer=200, stream=s)
        return st["x"]
    if st["what"] == "multirhs":
        st["mr"].apply_dev(st["nrhs"], st["U"], st["V"], s)
        return st["V"]
    server, out = st["server"], {}
    ids = {server.submit(op, method, b, rtol=1e-10, inner_rtol=0.1 if method & IR_RELIABLE else 1e-2, max_outer=200): k
           for k, (op, method, b) in enumerate(st["jobs"])}
    while len(out) < len(ids):
        server.step(8)
        for jid in server.poll():
            k = ids[jid]
            out[k] = server.result(jid, st["jobs"][k][2].size)[0]
    return [out[k] for k in range(len(ids))]


# ------------------------------------------------------------------ floors
def _counts(kind: str, n: int, ny: int = 0, nz: int = 0) -> tuple[int, int]:
    """(elements, DoFs)"""
    ny, nz = ny or n, nz or n
    c, e = (n + 1) * (ny + 1) * (nz + 1), n * ny * nz
    if kind == "hex8":
        return e, c
    edges = n * (ny + 1) * (nz + 1) + (n + 1) * ny * (nz + 1) + (n + 1) * (ny + 1) * nz
    if kind == "hex20":
        return e, 3 * (c + edges)
    return 6 * e, (2 * n + 1) ** 3


def _product(case: dict) -> tuple[float, float, int]:
    """Bytes and flops of one operator application, and the DoF count.  Each
    input once: the element map; the stored matrices (the upper triangles where
    an element has its own), or a factor per element, or its coordinates; u and v."""
    kind = case["mesh"]
    e, d = _counts(kind, case["n"], case.get("ny", 0), case.get("nz", 0))
    n, ks = DOFS[kind], {"fp64": 8, "fp32": 4, "bf16": 2}[case.get("prec", "fp64")]
    vs = 8 if ks == 8 else 4
    if case["what"] == "method2":
        nodes = 8 if kind == "hex8" else 20 if kind == "hex20" else 10
        pts = case["ngt"] ** 3
        per, fl = vs * d / (3 if kind == "hex20" else 1) * 3 / e + vs, pts * (1260 if kind == "hex20" else 30 * nodes + 85)
    elif case.get("matrices", "distinct" if kind == "tet10" else "scaled") == "scaled":
        per, fl = 8.0, 2 * n * n
    else:
        per, fl = ks * n * (n + 1) // 2, 2 * n * n
    return e * (per + 4 * n) + 2 * vs * d, e * fl, d


def _solve_work(case: dict) -> tuple[float, float]:
    """Iterations of Jacobi-CG to 1e-10 grow with n (2.4 n hex8, 60 n hex20, 10.6 n
    tet10); each is a product and the five vectors read and three written."""
    its = case["n"] * {"hex8": 2.4, "hex20": 60.0, "tet10": 10.6}[case["mesh"]]
    low = case["method"][:4]
    b, f, d = _product({**case, "prec": low})
    return its * (b + 8 * d * (8 if low == "fp64" else 4)), its * (f + 12 * d)


def work(case: dict) -> dict:
    if case["what"] in ("matvec", "method2"):
        b, f, _ = _product(case)
    elif case["what"] == "solve":
        b, f = _solve_work(case)
    elif case["what"] == "multirhs":
        b = f = 0.0
        for kind, dims in (("hex20", (case["n"], 0, 0)), ("hex8", (case["hx"], case["hy"], case["hz"]))):
            e, d = _counts(kind, *dims)
            b += e * (4 * DOFS[kind] + 8) + 8 * d * case["nrhs"]
            f += 2 * e * DOFS[kind] ** 2 * case["nrhs"]
    else:
        parts = [_solve_work(r) for r in _requests(case)]
        b, f = sum(x for x, _ in parts), sum(x for _, x in parts)
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ in 64 bits
def _reference_points(kind: str, ngt: int) -> list[tuple[np.ndarray, float]]:
    """(dN/dxi (nodes, 3), weight) at the quadrature points, from the shape functions."""
    x1, w1 = np.polynomial.legendre.leggauss(ngt)
    out = []
    for i in range(ngt):
        for j in range(ngt):
            for k in range(ngt):
                p, w = np.array([x1[i], x1[j], x1[k]]), w1[i] * w1[j] * w1[k]
                if kind == "tet10":  # the cube collapsed onto the tetrahedron, towards vertex 0
                    a, b, c = (1 + p) / 2
                    xi = np.array([a * b * c, a * b * (1 - c), a * (1 - b)])
                    w *= a * a * b / 8
                    L = np.array([1 - xi.sum(), *xi])
                    g = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
                    dn = [(4 * L[v] - 1) * g[v] for v in range(4)]
                    dn += [4 * (L[u] * g[v] + L[v] * g[u]) for u, v in ((0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3))]
                else:
                    dn = []
                    for c in _HEX_NODES[:20 if kind == "hex20" else 8]:
                        c = np.array(c, dtype=float)
                        f, df = 1 + c * p, c.copy()  # factors (1 + c x), and 1 - x^2 on the edge axis
                        f[c == 0], df[c == 0] = 1 - p[c == 0] ** 2, -2 * p[c == 0]
                        prod = [f[1] * f[2], f[0] * f[2], f[0] * f[1]]
                        if kind == "hex8":
                            dn.append([df[d] * prod[d] / 8 for d in range(3)])
                        elif (c == 0).any():
                            dn.append([df[d] * prod[d] / 4 for d in range(3)])
                        else:
                            t = c @ p - 2
                            dn.append([(df[d] * prod[d] * t + f.prod() * c[d]) / 8 for d in range(3)])
                out.append((np.array(dn), w))
    return out


_HEX_NODES = [(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1),
              (0, -1, -1), (1, 0, -1), (0, 1, -1), (-1, 0, -1), (0, -1, 1), (1, 0, 1), (0, 1, 1), (-1, 0, 1),
              (-1, -1, 0), (1, -1, 0), (1, 1, 0), (-1, 1, 0)]


def _method2_rows(case: dict, p: problems.Problem, seed: int, ue: np.ndarray, diag: bool = False) -> np.ndarray:
    """K_e u_e (or diag K_e) of every element from its coordinates."""
    x, s = _coords(case, p, seed), _scales(case, p, seed)
    nu = p.free.get("nu", 0.3)
    lam, mu = nu / ((1 + nu) * (1 - 2 * nu)), 0.5 / (1 + nu)
    out = np.zeros_like(ue)
    for lo in range(0, len(x), 1 << 15):
        sl = slice(lo, lo + (1 << 15))
        xe, u = x[sl], ue[sl].reshape(len(x[sl]), x.shape[1], -1)
        f = np.zeros_like(u)
        for dn, w in _reference_points(case["mesh"], case["ngt"]):
            J = xe.transpose(0, 2, 1) @ dn                # J[k][d] = dx_k / dxi_d
            g = dn @ np.linalg.inv(J)                     # dN/dx
            wq = (np.linalg.det(J) * w * s[sl])[:, None, None]
            if diag:
                gg = (g * g).sum(axis=2, keepdims=True)
                f += wq * (gg if u.shape[2] == 1 else (lam + mu) * g * g + mu * gg)
                continue
            H = u.transpose(0, 2, 1) @ g                  # du_i / dx_k
            if u.shape[2] == 3:
                e = H + H.transpose(0, 2, 1)
                H = mu * e + lam * np.trace(H, axis1=1, axis2=2)[:, None, None] * np.eye(3)
            f += wq * (g @ H.transpose(0, 2, 1))
        out[sl] = f.reshape(len(f), -1)
    return out


def _apply64(rows, p: problems.Problem, bc: str, diag):
    """u -> v in 64 bits; rows(ue) forms K_e u_e of all elements, diag() their diagonals."""
    gm = p.gmap.astype(np.int64)
    c = p.constrained.astype(np.int64)
    K_cc = np.bincount(gm.reshape(-1), weights=diag().reshape(-1), minlength=p.n_dofs)[c] if bc == "penalty" else None

    def f(u):
        w = u
        if bc == "identity":
            w = u.copy()
            w[c] = 0.0
        v = np.bincount(gm.reshape(-1), weights=rows(w[gm]).reshape(-1), minlength=p.n_dofs)
        if bc == "identity":
            v[c] = u[c]
        elif bc == "penalty":
            v[c] += (PENALTY - K_cc) * u[c]
        return v
    return f


def _stored64(case: dict, p: problems.Problem, seed: int):
    """(rows, diag) of _apply64 for element matrices."""
    s = _scales(case, p, seed)[:, None]
    if case.get("matrices", "distinct" if case["mesh"] == "tet10" else "scaled") == "scaled":
        return (lambda ue: s * (ue @ p.k_ref.T)), (lambda: s * np.diag(p.k_ref))
    K = _matrices(case, p, seed)
    return (lambda ue: (K @ ue[:, :, None])[:, :, 0]), (lambda: np.diagonal(K, axis1=1, axis2=2))


def _solve64(case: dict, seed: int):
    """Jacobi-CG in 64 bits to 1e-13; None where it would take long."""
    p = _of(case)
    if _solve_work(case)[1] > 6e10:
        return None
    rows, diag = _stored64(case, p, seed)
    A = _apply64(rows, p, "identity", diag)
    d = np.bincount(p.gmap.astype(np.int64).reshape(-1), weights=diag().reshape(-1), minlength=p.n_dofs)
    d[p.constrained.astype(np.int64)] = 1.0
    b = _rhs(p, seed)
    x, r = np.zeros_like(b), b.copy()
    z = r / d
    q, rz = z.copy(), r @ z
    for _ in range(20000):
        a = A(q)
        alpha = rz / (q @ a)
        x += alpha * q
        r -= alpha * a
        if r @ r <= 1e-26 * (b @ b):
            break
        z = r / d
        rz, old = r @ z, rz
        q = z + (rz / old) * q
    return x


def exact(case: dict, seed: int):
    if case["what"] in ("matvec", "method2"):
        p = _of(case)
        if case["what"] == "method2":
            rows, diag = (lambda ue: _method2_rows(case, p, seed, ue)), \
                (lambda: _method2_rows(case, p, seed, np.zeros(p.gmap.shape), diag=True))
        else:
            rows, diag = _stored64(case, p, seed)
        u = mesh.uniform(seed, 1, p.n_dofs, -1.0, 1.0)
        if case["prec"] != "fp64":
            u = u.astype(np.float32).astype(np.float64)
        return _apply64(rows, p, case["bc"], diag)(u)
    if case["what"] == "solve":
        return _solve64(case, seed)
    if case["what"] == "multirhs":
        out = []
        for p, s, U in _multirhs(case, seed):
            V, gm = torch.zeros(U.shape, dtype=torch.float64), torch.from_numpy(p.gmap.astype(np.int64))
            U64, K, sc = torch.from_numpy(U).double(), torch.from_numpy(p.k_ref), torch.from_numpy(s)
            for lo in range(0, len(gm), 4096):
                g = gm[lo:lo + 4096]
                ue = U64[g].transpose(0, 1).reshape(len(K), -1)
                rows = (K @ ue).view(len(K), len(g), -1) * sc[None, lo:lo + 4096, None]
                V.index_add_(0, g.t().reshape(-1), rows.view(-1, U.shape[1]))
            out.append(V.numpy())
        return out
    got = [_solve64(r, seed + i) if _solve_work(r)[1] < 1e10 else None for i, r in enumerate(_requests(case))]
    return got if any(g is not None for g in got) else None
