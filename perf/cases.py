"""Cases that time the framework through its public entry points.

Every case is a boundary-element problem like the ones the tests and the
benchmark use: icospheres (one, or several side by side, three radii apart)
of flat triangles with the 1/(4 pi r) centroid kernel, leaf size 20, eta 2
and ACA+ 1e-4 or 1e-5.  `mesh` names the subdivision of each sphere ("6+6":
two of 81,920 triangles); `cut` triangles are left out at the end, an open
surface with a size that is no multiple of anything.  The radius (0.5 to 2)
and the vectors (uniform in [-1, 1)) come from the seed.

What a case does in one pass (`path`):
  apply      Arena.apply: y = H x, FP64 factors, vectors on the device
  host       the reference-named product on host vectors: zau += H zu
  matmat     Arena.apply_block: Y = H X for k right-hand sides, FP64 factors
  bicgstab   Arena.bicgstab: an FP64 solve
  gcr_ir     gcr_ir: an FP64 solve refined over narrow factors
  multi      multi_gcr_ir: the same for several independent problems at once
  construct  DeviceHMatrix, its arena and the first product: mesh to result

Solves run to a residual of 1e-11, so that the solution is determined to
about as many digits and two solves can be compared.
"""
import importlib
import math

import numpy as np
import torch

SOLVE_EPS = 1e-11


def listed():
    return [
        # the smallest problem of the tests: launches and latency
        dict(name="apply-1k", path="apply", mesh="3", cut=0, eps=1e-4),
        # a small problem of an odd size
        dict(name="apply-6k", path="apply", mesh="4+3", cut=37, eps=1e-4),
        # the headline benchmark's product
        dict(name="apply-164k", path="apply", mesh="6+6", cut=0, eps=1e-5),
        # what a Fortran caller of the reference's interface gets per product
        dict(name="host-26k", path="host", mesh="5+4", cut=3, eps=1e-4),
        # several right-hand sides: few, an odd number, and the benchmark's 32 and 128
        dict(name="matmat-82k-k8", path="matmat", mesh="6", cut=0, eps=1e-5, k=8),
        dict(name="matmat-42k-k19", path="matmat", mesh="5+5+3", cut=5, eps=1e-4, k=19),
        dict(name="matmat-164k-k32", path="matmat", mesh="6+6", cut=0, eps=1e-5, k=32),
        dict(name="matmat-328k-k128", path="matmat", mesh="7", cut=0, eps=1e-5, k=128),
        # the tests' solve: short kernels, launch-bound
        dict(name="bicgstab-5k", path="bicgstab", mesh="4", cut=0, eps=1e-4),
        # mixed precision in earnest: narrow factors under FP64 refinement
        dict(name="gcr-ir-82k", path="gcr_ir", mesh="6", cut=0, eps=1e-5, low="bf16"),
        # the batch of uneven instances, narrow factors throughout
        dict(name="multi-gcr-59k", path="multi", mesh="5+5+4+4+4+3+3+2", cut=0, eps=1e-4,
             low="bf16_all"),
        # from a mesh to the first product
        dict(name="construct-82k", path="construct", mesh="6", cut=0, eps=1e-5),
    ]


# Largest mesh (triangles) that draw() takes for each path: at most the
# largest listed problem of that path.
_DRAW_MOST = {"apply": 163840, "host": 102400, "matmat": 327680, "bicgstab": 25600,
              "gcr_ir": 81920, "multi": 81920, "construct": 81920}


def _faces_of(mesh, cut=0):
    return sum(20 * 4 ** int(s) for s in mesh.split("+")) - cut


def draw(rng):
    path = rng.choice(["apply", "apply", "host", "matmat", "matmat", "matmat", "bicgstab",
                       "gcr_ir", "multi", "construct"])
    most = _DRAW_MOST[path]
    case = dict(path=path, eps=rng.choice([1e-4, 1e-5]))
    if path == "matmat":
        case["k"] = min(128, max(2, round(2 ** rng.uniform(1.0, 7.0))))
        most = min(most, 327680 * 128 // case["k"], 2 ** rng.uniform(13.0, 18.4))
    # spheres added largest first until a target size (uniform in its
    # logarithm) is met, at most eight
    target = min(most, 2 ** rng.uniform(10.0, math.log2(most)))
    parts, total = [], 0
    for s in (7, 6, 5, 4, 3, 2):
        size = 20 * 4 ** s
        while total + size <= target and len(parts) < 8:
            parts.append(s)
            total += size
            if path != "multi" and rng.random() < 0.5:
                break
    case["mesh"] = "+".join(str(s) for s in parts)
    case["cut"] = 0 if path == "multi" else rng.randint(1, max(2, total // 40))
    if path in ("gcr_ir", "multi"):
        case["low"] = rng.choice(["f32", "bf16", "bf16_all"])
    return case


# ---------------------------------------------------------------------------
# meshes and vectors (numpy only: exact() uses them too)
# ---------------------------------------------------------------------------
def _icosphere(subdiv):
    """Nodes and faces of the unit icosahedron subdivided `subdiv` times."""
    t = (1.0 + 5.0 ** 0.5) / 2.0
    v = np.array([(-1, t, 0), (1, t, 0), (-1, -t, 0), (1, -t, 0), (0, -1, t), (0, 1, t),
                  (0, -1, -t), (0, 1, -t), (t, 0, -1), (t, 0, 1), (-t, 0, -1), (-t, 0, 1)], float)
    v /= np.linalg.norm(v, axis=1)[:, None]
    f = np.array([(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9),
                  (5, 11, 4), (11, 10, 2), (10, 7, 6), (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6),
                  (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11), (6, 2, 10), (8, 6, 7), (9, 8, 1)])
    for _ in range(subdiv):
        e = np.stack([f, np.roll(f, -1, axis=1)], axis=2)  # (faces, 3 edges, 2 ends)
        e.sort(axis=2)
        key, at = np.unique(e[:, :, 0] * len(v) + e[:, :, 1], return_inverse=True)
        mid = v[key // len(v)] + v[key % len(v)]
        mid /= np.linalg.norm(mid, axis=1)[:, None]
        m = at.reshape(-1, 3) + len(v)
        v = np.vstack([v, mid])
        f = np.stack([np.stack([f[:, 0], m[:, 0], m[:, 2]], 1),
                      np.stack([f[:, 1], m[:, 1], m[:, 0]], 1),
                      np.stack([f[:, 2], m[:, 2], m[:, 1]], 1), m], 1).reshape(-1, 3)
    return v, f


_spheres = {}  # unit icospheres by subdivision: a program keeps its meshes


def _sphere(s):
    if s not in _spheres:
        _spheres[s] = _icosphere(s)
    return _spheres[s]


def _meshes(case, seed):
    """The case's spheres as a list of (nodes, faces), radius from the seed;
    the last `cut` faces left out."""
    rng = np.random.default_rng([seed, 1])
    out = []
    for i, s in enumerate(int(p) for p in case["mesh"].split("+")):
        v, f = _sphere(s)
        if i == 0 or case["path"] == "multi":
            r = rng.uniform(0.5, 2.0)
        x = 0.0 if case["path"] == "multi" else 3.0 * r * i
        out.append((r * v + np.array([x, 0.0, 0.0]), f))
    return out


def _mesh(case, seed):
    nodes, faces, off = [], [], 0
    for v, f in _meshes(case, seed):
        nodes.append(v)
        faces.append(f + off)
        off += len(v)
    faces = np.vstack(faces)
    return (np.ascontiguousarray(np.vstack(nodes)),
            np.ascontiguousarray(faces[:len(faces) - case["cut"]], dtype=np.int32))


def _vector(seed, n, k=1):
    """k interleaved vectors in the numbering of the faces, as (n, k)."""
    return np.random.default_rng([seed, 2]).uniform(-1.0, 1.0, (n, k))


# ---------------------------------------------------------------------------
# the framework
# ---------------------------------------------------------------------------
def _package():
    H = importlib.import_module("hacapk-magma_amd")
    if H.hmv_lib().hmv_init(0) != 0:
        raise RuntimeError(H.hmv_lib().hmv_last_error().decode())
    return H


def _device_matrix(H, case, seed):
    return H.DeviceHMatrix(*_mesh(case, seed), H.baseline_params(aca_eps=case["eps"]))


def prepare(case, seed):
    H = _package()
    path = case["path"]
    state = {"H": H, "path": path, "case": case}
    if path == "construct":
        nodes, faces = _mesh(case, seed)
        x = torch.from_numpy(_vector(seed, len(faces))[:, 0]).cuda()
        return dict(state, nodes=nodes, faces=faces, x=x)
    if path == "host":
        hm = H.HMatrix(*_mesh(case, seed), H.baseline_params(aca_eps=case["eps"]))
        lp = H.make_leafmtxp(hm)
        H.adot_body_lfcpy_batch_sorted(hm.nd, lp)
        zu = hm.to_cluster_order(_vector(seed, hm.nd)[:, 0])
        return dict(state, hm=hm, lp=_Bound(H, lp), zu=zu, zau=np.zeros(hm.nd))
    if path == "multi":
        hms = [H.HMatrix(v, np.ascontiguousarray(f, np.int32), H.baseline_params(aca_eps=case["eps"]))
               for v, f in _meshes(case, seed)]
        b = _vector(seed, sum(hm.nd for hm in hms))[:, 0]
        off = np.cumsum([0] + [hm.nd for hm in hms])
        b = np.concatenate([hm.to_cluster_order(b[o:o + hm.nd]) for hm, o in zip(hms, off)])
        return dict(state, a64=H.MultiArena(hms, "f64"), low=H.MultiArena(hms, case["low"]), b=b)
    dm = _device_matrix(H, case, seed)
    state["a64"] = dm.arena("f64")
    if path == "gcr_ir":
        state["low"] = dm.arena(case["low"])
    v = _vector(seed, dm.nd, case.get("k", 1))[dm.lod - 1]
    dm.free()
    if path in ("bicgstab", "gcr_ir"):
        state["b"] = np.ascontiguousarray(v[:, 0])
    else:
        state["x"] = torch.from_numpy(np.ascontiguousarray(v)).cuda()
        state["y"] = torch.zeros_like(state["x"])
    return state


class _Bound:
    """A container the reference-named calls hold an arena for, given back
    when the state goes."""

    def __init__(self, H, lp):
        self.H, self.lp = H, lp

    def __del__(self):
        self.H.adot_body_lfdel_batch(self.lp)


def run(state):
    H, path = state["H"], state["path"]
    if path == "apply":
        stream = torch.cuda.current_stream().cuda_stream
        state["a64"].apply(state["x"].data_ptr(), state["y"].data_ptr(), stream=stream)
        return state["y"]
    if path == "matmat":
        stream = torch.cuda.current_stream().cuda_stream
        state["a64"].apply_block(state["x"].data_ptr(), state["y"].data_ptr(),
                                 state["x"].shape[1], stream=stream)
        return state["y"]
    if path == "host":
        zau = state["zau"]
        zau[:] = 0.0
        H.adot_body_lfmtx_batch(zau, state["lp"].lp, state["zu"])
        return zau
    if path == "bicgstab":
        return state["a64"].bicgstab(state["b"], eps=SOLVE_EPS, maxit=500, check_every=8,
                                     history=False)[0]
    if path == "gcr_ir":
        return H.gcr_ir(state["a64"], state["low"], state["b"], eps=SOLVE_EPS)[0]
    if path == "multi":
        return H.multi_gcr_ir(state["a64"], state["low"], state["b"], eps=SOLVE_EPS)[0]
    # construct: the user's numbering in and out
    dm = H.DeviceHMatrix(state["nodes"], state["faces"],
                         H.baseline_params(aca_eps=state["case"]["eps"]))
    a = dm.arena("f64")
    lod = torch.from_numpy(dm.lod - 1).cuda()
    x = state["x"][lod]
    y = torch.empty_like(x)
    a.apply(x.data_ptr(), y.data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
    out = torch.empty_like(y)
    out[lod] = y
    kt = dm.kt
    torch.cuda.current_stream().synchronize()  # before the arena goes
    a.free()
    dm.free()
    return {"y": out, "ranks": kt}


def work(case):
    """Bytes and flops of one pass.  E: entries of the dense blocks and the
    low-rank factors.  A product reads them once (8 bytes each; the narrow
    copies 2 or 4) with the vectors; a solve needs about as many products as
    its method took when the cases were chosen; a construction evaluates and
    writes the factors once and lays them out once (one read, one write)."""
    H = _package()
    if case["path"] == "multi":
        p = H.baseline_params(aca_eps=case["eps"])
        tables = [H.HMatrix(v, np.ascontiguousarray(f, np.int32), p).leaf_table()
                  for v, f in _meshes(case, 0)]
        t = np.vstack(tables)
    else:
        dm = _device_matrix(H, case, 0)
        t = dm.table.copy()
        dm.free()
    lt, kt, ndl, ndt = t[:, 0], t[:, 1], t[:, 3], t[:, 5]
    lr, dense = int((kt * (ndl + ndt))[lt == 1].sum()), int((ndl * ndt)[lt == 2].sum())
    n, e, k = _faces_of(case["mesh"], case["cut"]), lr + dense, case.get("k", 1)
    if case["path"] in ("apply", "matmat", "host"):
        return {"bytes": 8.0 * e + 16.0 * n * k, "flops": 2.0 * e * k}
    if case["path"] == "construct":
        return {"bytes": 32.0 * e + 16.0 * n, "flops": 12.0 * e}
    if case["path"] == "bicgstab":
        products = 60
        return {"bytes": products * (8.0 * e + 48.0 * n), "flops": products * 2.0 * e}
    low = {"f32": 4.0 * e, "bf16": 2.0 * lr + 4.0 * dense, "bf16_all": 2.0 * e}[case["low"]]
    inner, outer = 110, 6
    return {"bytes": inner * (low + 48.0 * n) + outer * (8.0 * e + 48.0 * n),
            "flops": (inner + outer) * 2.0 * e}


# ---------------------------------------------------------------------------
# the same in 64 bits, without the framework: the dense matrix instead of its
# H-matrix (they differ by the ACA tolerance)
# ---------------------------------------------------------------------------
def _cluster_order(cent, leaf=20):
    """The cluster tree's numbering: boxes are halved along their longest
    side until at most `leaf` points are left; the points on the wrong side
    change places, first with last."""
    order = np.arange(len(cent))
    todo = [(0, len(cent))]
    while todo:
        lo, hi = todo.pop()
        if hi - lo <= leaf:
            continue
        p = cent[order[lo:hi]]
        a, b = p.min(axis=0), p.max(axis=0)
        d = int(np.argmax(b - a))
        up = p[:, d] > (b[d] + a[d]) / 2
        c = int(len(up) - up.sum())
        left = lo + np.nonzero(up[:c])[0]
        right = (lo + c + np.nonzero(~up[c:])[0])[::-1]
        order[left], order[right] = order[right], order[left].copy()
        todo += [(lo, lo + c), (lo + c, hi)]
    return order


def _self_terms(tri, cent):
    """Integral of 1/|c - y| over each triangle, c its centre: the sum over
    the edges of h ln((r_b + t_b) / (r_a + t_a)), h the centre's distance from
    the edge's line, r and t the end points' distances from c and along it."""
    s = np.zeros(len(tri))
    for i in range(3):
        a, b = tri[:, i] - cent, tri[:, (i + 1) % 3] - cent
        e = b - a
        e /= np.linalg.norm(e, axis=1)[:, None]
        ra, rb = np.linalg.norm(a, axis=1), np.linalg.norm(b, axis=1)
        ta, tb = (a * e).sum(1), (b * e).sum(1)
        h = np.linalg.norm(a - ta[:, None] * e, axis=1)
        s += h * np.log((rb + tb) / (ra + ta))
    return s


def _dense(nodes, faces):
    """Order, centres, areas and diagonal of the dense matrix."""
    tri = nodes[faces]
    cent = (tri[:, 0] + tri[:, 1] + tri[:, 2]) / 3.0
    area = 0.5 * np.linalg.norm(np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]), axis=1)
    return _cluster_order(cent), cent, area, _self_terms(tri, cent) / (4.0 * math.pi)


def _rows(cent, area, diag, lo, hi):
    """Rows lo..hi of the dense matrix (torch, 64 bits)."""
    d2 = torch.zeros(hi - lo, len(area), dtype=torch.float64, device=cent.device)
    for c in range(3):
        d2 += (cent[lo:hi, c, None] - cent[None, :, c]).square_()
    at = torch.arange(lo, hi, device=cent.device)
    d2[at - lo, at] = 1.0
    m = (area / (4.0 * math.pi))[None, :] * d2.rsqrt_()
    m[at - lo, at] = diag[lo:hi]
    return m


def exact(case, seed):
    path = case["path"]
    n = _faces_of(case["mesh"], case["cut"])
    if path == "multi" or (path in ("bicgstab", "gcr_ir") and n > 8192):
        return None  # a dense solve of this size takes too long
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    order, cent, area, diag = _dense(*_mesh(case, seed))
    if path == "construct":
        order = np.arange(n)
    x = torch.from_numpy(_vector(seed, n, case.get("k", 1))[order]).to(dev)
    c, a, d = (torch.from_numpy(np.ascontiguousarray(v[order])).to(dev) for v in (cent, area, diag))
    if path in ("bicgstab", "gcr_ir"):
        m = _rows(c, a, d, 0, n).cpu().numpy()
        return np.linalg.solve(m, x[:, 0].cpu().numpy())
    step = max(1, min(n, 2 ** 28 // n))
    y = torch.cat([_rows(c, a, d, i, min(n, i + step)) @ x for i in range(0, n, step)])
    if path == "host":
        return y[:, 0].cpu().numpy()
    if path == "construct":
        return {"y": y[:, 0], "ranks": None}
    return y
