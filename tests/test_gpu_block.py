"""Multi-right-hand-side H-matmat (vector units for few right-hand sides,
MFMA for more) and block BiCGSTAB through the C ABI.

Bar: every column of the H-matmat equals the single-vector apply of that
column (FP64: <= 1e-13 relative, FP32 / BF16 arenas: <= 1e-5 relative, both
accumulate in FP32 but in different orders) and the CPU oracle (FP64 <= 1e-12);
block BiCGSTAB columns reach the true residual bar and agree with the
single-vector solver's solutions.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("k", [1, 3, 8, 16, 32, 40, 64, 72, 128])
def test_matmat_f64_columns(gpu, O, two_spheres4, k):
    hm = two_spheres4
    a = gpu.Arena(hm, "f64")
    X = np.stack([gpu.uniform(100 + j, hm.nd) for j in range(k)], axis=1)
    Y = a.matmat(X)
    worst = 0.0
    for j in sorted({0, k // 2, k - 1}):
        y1 = a.matvec(X[:, j])
        worst = max(worst, _rel(Y[:, j], y1))
        assert _rel(Y[:, j], O.adot_body_lfmtx(hm, X[:, j])) <= 1e-12
    print("k", k, "max rel diff vs single apply %.2e" % worst, flush=True)
    assert worst <= 1e-13
    a.free()


@pytest.mark.parametrize("prec,k", [("f32", 8), ("f32", 32), ("bf16", 16), ("bf16_all", 8),
                                    ("f32", 4), ("bf16", 2), ("bf16_all", 3), ("f32", 128),
                                    ("bf16_all", 72)])
def test_matmat_low_precision(gpu, O, two_spheres4, prec, k):
    """Narrow arenas: k <= 4 runs on the vector units (hmv_kstream.hip),
    larger k on FP32 MFMAs (two 16-row tiles per wave above k = 64)."""
    hm = two_spheres4
    a = gpu.Arena(hm, prec)
    X = np.stack([gpu.uniform(200 + j, hm.nd) for j in range(k)], axis=1)
    Y = a.matmat(X)
    for j in (0, k - 1):
        assert _rel(Y[:, j], a.matvec(X[:, j])) <= 1e-5
        assert _rel(Y[:, j], O.adot_body_lfmtx(hm, X[:, j])) <= {"f32": 1e-5, "bf16": 2e-2, "bf16_all": 2e-2}[prec]
    a.free()


TOL = {"f64": 1e-12, "f32": 1e-5, "bf16": 2e-2, "bf16_all": 2e-2}


def _paths(prec, k):
    """Every H-matmat path choice of k's classes: (vector, tiles per unit)."""
    vec_max = 8 if prec == "f64" else 4
    kt = (k + 15) // 16
    tiles = [4, 2] if kt == 1 else [2, 1] if kt <= 4 else ([1, 2] if prec == "f64" else [2, 1])
    out = [(1, tiles[0])] if k <= vec_max else []
    return out + [(0, t) for t in tiles]


@pytest.mark.parametrize("prec,k", [("f64", 3), ("f64", 8), ("f64", 16), ("f64", 40), ("f64", 128),
                                    ("f32", 4), ("f32", 72), ("bf16_all", 128)])
def test_matmat_every_path(gpu, O, two_spheres4, prec, k):
    """Each path the block tuning can select (vector units, MFMA with each
    instantiated tiles-per-unit width) gives the oracle's product; the
    arena reports the path it was set to."""
    hm = two_spheres4
    a = gpu.Arena(hm, prec)
    X = np.stack([gpu.uniform(300 + j, hm.nd) for j in range(k)], axis=1)
    for vec, tiles in _paths(prec, k):
        a.set_block_tuning(k, vec, tiles)
        assert a.block_tuning(k) == {"vector": vec, "tiles_per_unit": tiles}
        Y = a.matmat(X)
        for j in (0, k - 1):
            assert _rel(Y[:, j], O.adot_body_lfmtx(hm, X[:, j])) <= TOL[prec], (vec, tiles, j)
    a.free()


@pytest.mark.parametrize("prec,k", [("f64", 7), ("f64", 8), ("f64", 64), ("f64", 128),
                                    ("f32", 128)])
def test_matmat_inputs_at_any_alignment(gpu, sphere4, prec, k):
    """Inputs that start 8 bytes past a 16-byte boundary (a caller's x may
    start anywhere) take the paths that read inputs one value at a time
    instead of in 16-byte pairs; the product is bit-equal to the aligned
    one (the same values reach the same FMAs), and odd k uses the unpaired
    staging too."""
    a = gpu.Arena(sphere4, prec)
    X = np.stack([gpu.uniform(700 + j, sphere4.nd) for j in range(k)], axis=1)
    Y_al = a.matmat(X)
    buf = gpu.DeviceBuffer.from_array(np.concatenate([[0.0], X.reshape(-1)]))
    dy = gpu.DeviceBuffer.from_array(np.zeros(X.size))
    a.apply_block(buf.ptr + 8, dy.ptr, k)
    assert np.array_equal(dy.download().reshape(sphere4.nd, k), Y_al)
    buf.free()
    dy.free()
    a.free()


@pytest.mark.parametrize("prec,k", [("f64", 8), ("f64", 32), ("f32", 4)])
def test_block_autotune(gpu, O, sphere4, prec, k):
    """hmv_autotune_block sets the fastest path of k's classes: no slower
    than the defaults, reported back by the arena, and its product matches
    the oracle."""
    a = gpu.Arena(sphere4, prec)
    dflt = a.block_tuning(k)
    best, best_ms, dflt_ms = a.autotune_block(k, reps=3)
    print(prec, k, "default", dflt, "best", best, "%.4f ms (default %.4f ms)" % (best_ms, dflt_ms),
          flush=True)
    assert 0 < best_ms <= dflt_ms
    assert a.block_tuning(k) == best
    X = np.stack([gpu.uniform(400 + j, sphere4.nd) for j in range(k)], axis=1)
    Y = a.matmat(X)
    assert _rel(Y[:, k - 1], O.adot_body_lfmtx(sphere4, X[:, k - 1])) <= TOL[prec]
    a.free()


def test_block_tuning_rejects(gpu, sphere3):
    a, n = gpu.Arena(sphere3, "f64"), gpu.Arena(sphere3, "f32")
    with pytest.raises(gpu.HmvError, match="vector path"):
        a.set_block_tuning(16, 1)
    with pytest.raises(gpu.HmvError, match="vector path"):
        n.set_block_tuning(8, 1)
    with pytest.raises(gpu.HmvError, match="tiles_per_unit"):
        a.set_block_tuning(32, 0, 4)
    with pytest.raises(gpu.HmvError):
        a.block_tuning(129)
    a.free()
    n.free()


def test_matmat_beta_accumulates(gpu, sphere4):
    a = gpu.Arena(sphere4, "f64")
    k = 8
    X = np.stack([gpu.uniform(300 + j, sphere4.nd) for j in range(k)], axis=1)
    Y0 = np.stack([gpu.uniform(400 + j, sphere4.nd) for j in range(k)], axis=1)
    dx, dy = gpu.DeviceBuffer.from_array(X.reshape(-1)), gpu.DeviceBuffer.from_array(Y0.reshape(-1))
    a.apply_block(dx.ptr, dy.ptr, k, beta=1.0)
    gpu.hmv_lib().hmv_device_synchronize()
    Y = dy.download().reshape(sphere4.nd, k)
    assert _rel(Y, Y0 + a.matmat(X)) <= 1e-13
    a.free()


def test_block_bicgstab_matches_single(gpu, sphere4):
    hm = sphere4
    a = gpu.Arena(hm, "f64")
    k = 8
    B = np.stack([gpu.uniform(500 + j, hm.nd) for j in range(k)], axis=1)
    B[:, 0] = 1.0
    U, cols, info = a.block_bicgstab(B, eps=1e-8, maxit=500, check_every=4)
    print("block", info, [c["nstp"] for c in cols], flush=True)
    assert info["status_name"] == "converged"
    for j in range(k):
        assert cols[j]["status_name"] == "converged" and cols[j]["true_relres"] < 1e-8 * 1.5
        u1, i1, _ = a.bicgstab(B[:, j], eps=1e-8, maxit=500)
        assert abs(cols[j]["nstp"] - i1["nstp"]) <= 3
        assert _rel(U[:, j], u1) < 1e-6
    a.free()


def test_block_bicgstab_stops_columns_independently(gpu, sphere4):
    """A zero right-hand side stops its column at setup (non-finite relative
    residual); the other columns still converge."""
    hm = sphere4
    a = gpu.Arena(hm, "f64")
    B = np.stack([gpu.uniform(600 + j, hm.nd) for j in range(4)], axis=1)
    B[:, 2] = 0.0
    U, cols, info = a.block_bicgstab(B, eps=1e-8, maxit=500)
    assert cols[2]["status_name"] == "nonfinite" and cols[2]["nstp"] == 0
    assert np.all(U[:, 2] == 0.0)
    for j in (0, 1, 3):
        assert cols[j]["status_name"] == "converged"
    a.free()


def test_block_rejects_bad_k(gpu, sphere3):
    a = gpu.Arena(sphere3, "f64")
    with pytest.raises(gpu.HmvError):
        a.block_bicgstab(np.ones((sphere3.nd, 3)))
    with pytest.raises(gpu.HmvError):
        a.matmat(np.ones((sphere3.nd, 129)))
    a.free()


@pytest.mark.parametrize("prec,inner", [("f32", 1e-4), ("bf16", 1e-2)])
def test_block_refinement(gpu, O, sphere4, prec, inner):
    """hmv_block_bicgstab_ir: FP64 block residuals on the FP64 arena, inner
    block BiCGSTAB on the low-precision arena; every column reaches a true
    1e-8 (recomputed by the oracle) and the single FP64 solve's solution
    within cond * 2e-8 (cond = 2 sqrt(N) + 1, the sphere single-layer
    operator's eigenvalue spread); a zero column stops at once."""
    hm = sphere4
    a64, alow = gpu.Arena(hm, "f64"), gpu.Arena(hm, prec)
    k = 8
    B = np.stack([gpu.uniform(700 + j, hm.nd) for j in range(k)], axis=1)
    B[:, 1] = 1.0
    B[:, 5] = 0.0
    U, cols, info = gpu.block_bicgstab_ir(a64, alow, B, eps=1e-8, inner_eps=inner, max_outer=30,
                                          max_inner=500)
    print(prec, info, [(c["nstp"], "%.1e" % c["true_relres"]) for c in cols], flush=True)
    assert info["outer"] >= 2
    assert cols[5]["status_name"] == "nonfinite" and cols[5]["nstp"] == 0
    assert np.all(U[:, 5] == 0.0)
    bound = (2.0 * np.sqrt(hm.nd) + 1.0) * 2e-8
    for j in range(k):
        if j == 5:
            continue
        tr = _rel(O.adot_body_lfmtx(hm, U[:, j]), B[:, j])
        assert cols[j]["status_name"] == "converged" and tr < 1e-8
        u1, i1, _ = a64.bicgstab(B[:, j], eps=1e-8, maxit=500)
        assert _rel(U[:, j], u1) < bound
    a64.free()
    alow.free()


@pytest.mark.parametrize("prec", ["f64", "f32", "bf16", "bf16_all"])
@pytest.mark.parametrize("k", [9, 16, 32, 40, 64, 128])
def test_matmat_waves_sharing_a_unit(gpu, O, prec, k):
    """Launches of few units share each unit's columns among several waves:
    blocks from one column to a few past two windows of 1,024, and of one to
    several 16-row tiles, against the oracle."""
    from synthetic_leaves import LeafSet
    nd = 5000
    cols = [1, 3, 4, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 255, 500, 1023, 1024, 1025, 1040,
            1088, 2047, 2048, 2049, 2113]
    lv, r = [], 0
    for i, nc in enumerate(cols):
        rows = [1, 15, 16, 17, 33, 48, 70][i % 7]
        lv.append(("dense", r, rows, 7 * i, nc, 0))
        if i % 3 == 0:
            lv.append(("lowrank", r, rows, 100 + i, 10 + 40 * i, 1 + i))
        r += rows
    hm = LeafSet(gpu, nd, lv, 4)
    a = gpu.Arena(hm, prec)
    X = np.stack([gpu.uniform(60 + j, nd) for j in range(k)], axis=1)
    Y = a.matmat(X)
    tol = {"f64": 1e-12, "f32": 1e-5, "bf16": 2e-2, "bf16_all": 2e-2}[prec]
    for j in sorted({0, k // 2, k - 1}):
        ref = O.adot_body_lfmtx(hm, X[:, j])
        assert np.linalg.norm(Y[:, j] - ref) / np.linalg.norm(ref) <= tol
    assert np.array_equal(a.matmat(X), Y)
    a.free()


@pytest.fixture(scope="module")
def sphere6_arenas(gpu):
    nodes, faces = gpu.icosphere(6)  # more units than share waves
    dm = gpu.DeviceHMatrix(nodes, faces, gpu.baseline_params(aca_eps=1e-4))
    out = {p: dm.arena(p) for p in ("f64", "bf16")}
    dm.free()
    yield out
    for a in out.values():
        a.free()


@pytest.mark.parametrize("prec", ["f64", "bf16"])
@pytest.mark.parametrize("k", [17, 18, 31, 33, 47, 62, 63, 65, 97, 126, 127])
def test_matmat_pairs_up_to_the_last_column(gpu, sphere4, sphere6_arenas, prec, k):
    """A lane reads pairs of right-hand sides; with k odd the last pair starts
    one column early.  Every column has the bits it has among a full tile
    count of right-hand sides (the others' inputs do not enter its sums)."""
    full = 32 if k <= 32 else 64 if k <= 64 else 128
    small = gpu.Arena(sphere4, prec)
    for a in (small, sphere6_arenas[prec]):
        X = gpu.uniform(k, a.nd * full).reshape(a.nd, full)
        ref = a.matmat(X)[:, :k]
        assert np.array_equal(a.matmat(np.ascontiguousarray(X[:, :k])), ref)
    small.free()


# a pair of tiles reads rows in twos: row counts from one tile to beyond a
# group of four, odd ones with a row on its own at the end of the block
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16", "bf16_all"])
def test_matmat_pairs_of_rows(gpu, prec):
    """Every row of every column within the rounding of its storage (2^-8 for
    BF16 factors, twice for a low-rank product of two, 2^-23 and 2^-52 terms
    for the others and for up to 130 summed columns) of sum |a| |x|: an entry
    missed or read twice is a tenth of that sum and more."""
    from synthetic_leaves import LeafSet
    rows = [1, 15, 16, 17, 18, 19, 23, 31, 32, 33, 34, 47, 48, 49, 63, 64, 65, 79, 127, 129]
    nd, lv, r = 2048, [], 0
    for i, nr in enumerate(rows):
        lv.append(("dense", r, nr, 30 * i, 1 + i % 9, 0))
        # a rank of nr: the rows of a phase-1 item
        lv.append(("lowrank", r, nr, 1000 + 40 * i, 1 + (5 * i) % 9, nr))
        r += nr
    lv.append(("dense", 2017, 31, 2000, 7, 0))  # the last block
    hm = LeafSet(gpu, nd, lv, 4)
    A, S = np.zeros((nd, nd)), np.zeros((nd, nd))
    for (kind, r0, nr, c0, nc, q), buf in zip(lv, hm._bufs):
        if kind == "dense":
            M = buf.reshape(nr, nc)
            A[r0:r0 + nr, c0:c0 + nc] += M
            S[r0:r0 + nr, c0:c0 + nc] += np.abs(M)
        else:
            V, U = buf[:nc * q].reshape(q, nc), buf[nc * q:].reshape(q, nr)
            A[r0:r0 + nr, c0:c0 + nc] += U.T @ V
            S[r0:r0 + nr, c0:c0 + nc] += np.abs(U).T @ np.abs(V)
    eps = {"f64": 140 * 2.0 ** -52, "f32": 140 * 2.0 ** -23}.get(prec, 2.0 ** -7 + 140 * 2.0 ** -23)
    a = gpu.Arena(hm, prec)
    for k in (9, 16, 19, 32, 50, 64, 128):
        X = gpu.uniform(k, nd * k).reshape(nd, k)
        Y = a.matmat(X)
        assert np.all(np.abs(Y - A @ X) <= eps * (S @ np.abs(X))), k
    a.free()
