"""Device construction (hmv_construct): dense entries and ACA+ on the GPU
against the host fill (the restatement of HACApK_generate's fill,
m_HACApK_base.f90:783-1051), and arenas repacked from device factors against
arenas from host factors."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _leaf_values(hm, lod):
    """Per leaf: (ltmtx, factors, diagonal mask or None)."""
    out = []
    for r in hm.leaves():
        if r.ltmtx == 1:
            n = (r.ndt + r.ndl) * r.kt
            out.append((1, np.ctypeslib.as_array(r.a1, shape=(n,)).copy() if n else np.zeros(0), None))
        else:
            a = np.ctypeslib.as_array(r.a1, shape=(r.ndl, r.ndt)).copy()
            rows = lod[r.nstrtl - 1:r.nstrtl - 1 + r.ndl]
            cols = lod[r.nstrtt - 1:r.nstrtt - 1 + r.ndt]
            out.append((2, a, rows[:, None] == cols[None, :]))
    return out


def test_centroid_kernel_fill_matches_host(gpu, O, H):
    """With the centroid kernel an off-diagonal entry is one sqrt and one
    division, correctly rounded on either side, and ACA+ runs the same
    arithmetic in the same order: ranks, every low-rank factor and every
    off-diagonal dense entry equal the host fill's bit for bit.  The diagonal
    (the analytic self term, through atan2 and log) may differ by an ulp."""
    nodes, faces = H.icosphere(4)
    p = H.baseline_params(aca_eps=1e-5)
    host = H.HMatrix(nodes, faces, p)
    dev = H.DeviceHMatrix(nodes, faces, p)
    assert np.array_equal(dev.table, host.leaf_table())
    got = dev.download()
    ndiff = 0
    for (kind, x, diag), (_, y, _) in zip(_leaf_values(host, host.lod), _leaf_values(got, host.lod)):
        if kind == 1:
            assert np.array_equal(x, y)
        else:
            assert np.array_equal(x[~diag], y[~diag])
            assert np.all(np.abs(x[diag] - y[diag]) <= 4e-16 * np.abs(x[diag]))
            ndiff += int((x[diag] != y[diag]).sum())
    print("leaves", host.nlf, "diagonal entries differing by an ulp:", ndiff,
          "device fill %.4f s" % dev.fill_seconds, flush=True)
    x = H.uniform(3, host.nd)
    y, yr = O.adot_body_lfmtx(got, x), O.adot_body_lfmtx(host, x)
    assert np.linalg.norm(y - yr) / np.linalg.norm(yr) < 1e-15
    dev.free()


def test_analytic_kernel_fill(gpu, O, H):
    """The reference's own kernel (face_integral for every pair) through the
    device's atan2/log: entries differ from the host's in the last bits, which
    can change a near-tied ACA+ pivot; both fills approximate the same matrix
    to the ACA tolerance."""
    d = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                             "input_1ts_mesh.npz"))
    p = H.HParams(leaf_size=15, aca_eps=1e-6, kernel="ppohbem")
    host = H.HMatrix(d["nodes"], d["faces"], p)
    dev = H.DeviceHMatrix(d["nodes"], d["faces"], p)
    ht = host.leaf_table()
    assert np.array_equal(dev.table[:, [0, 2, 3, 4, 5]], ht[:, [0, 2, 3, 4, 5]])
    assert np.mean(dev.table[:, 1] != ht[:, 1]) < 0.02  # ranks
    got = dev.download()
    A = O.dense(host)
    x = H.uniform(4, host.nd)
    ya = A @ x
    for hm in (host, got):
        assert np.linalg.norm(O.adot_body_lfmtx(hm, x) - ya) / np.linalg.norm(ya) < 2e-5
    dense_dev = O.dense(got)
    assert np.linalg.norm(dense_dev - A) / np.linalg.norm(A) < 2e-5
    dev.free()


def test_high_rank_blocks_take_the_second_pass(gpu, O, H):
    """ACA+ to 1e-14 needs more columns than the first pass reserves (64) on
    the larger blocks; those blocks run again with their full bound and
    still equal the host fill."""
    nodes, faces = H.icosphere(4)
    p = H.baseline_params(aca_eps=1e-14)
    host = H.HMatrix(nodes, faces, p)
    dev = H.DeviceHMatrix(nodes, faces, p)
    assert dev.kt.max() > 64
    assert np.array_equal(dev.table, host.leaf_table())
    got = dev.download()
    for (kind, x, diag), (_, y, _) in zip(_leaf_values(host, host.lod), _leaf_values(got, host.lod)):
        if kind == 1:
            assert np.array_equal(x, y)
    dev.free()


@pytest.mark.parametrize("prec", ["f64", "f32", "bf16", "bf16_all"])
def test_arena_from_device_factors(gpu, O, H, tmp_path, prec):
    """The arena repacked on the device from device factors is byte-equal to
    the host repack of the same factors (downloaded), and applies bit-equal."""
    nodes, faces = H.icosphere(4)
    p = H.baseline_params(aca_eps=1e-5)
    dev = H.DeviceHMatrix(nodes, faces, p)
    got = dev.download()
    a = dev.arena(prec)
    b = H.Arena(got, prec)
    x = H.uniform(5, dev.nd)
    assert np.array_equal(a.matvec(x), b.matvec(x))
    a.save(tmp_path / "dev.hmv")
    b.save(tmp_path / "host.hmv")
    assert (tmp_path / "dev.hmv").read_bytes() == (tmp_path / "host.hmv").read_bytes()
    y = a.matvec(x)
    y_ref = O.adot_body_lfmtx(got, x)
    tol = {"f64": 1e-12, "f32": 1e-6, "bf16": 2e-2, "bf16_all": 2e-2}[prec]
    assert np.linalg.norm(y - y_ref) / np.linalg.norm(y_ref) < tol
    a.free()
    b.free()
    dev.free()


def _construct_blocks(H, nodes, faces, blocks, eps):
    """hmv_construct on low-rank blocks (first row, rows, first column,
    columns; 0-based, faces in their own order): [U V^T] per block and the
    dense matrix's entry function as an array of rows."""
    import ctypes as C
    rec = (H.LeafRec * len(blocks))()
    for r, (l0, ndl, t0, ndt) in zip(rec, blocks):
        r.ltmtx, r.nstrtl, r.ndl, r.nstrtt, r.ndt = 1, l0 + 1, ndl, t0 + 1, ndt
    tri = nodes[faces]
    cent = np.ascontiguousarray((tri[:, 0] + tri[:, 1] + tri[:, 2]) / 3.0)
    area = 0.5 * np.linalg.norm(np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]), axis=1)
    lod = np.arange(1, len(faces) + 1, dtype=np.int32)
    cp = H._ConstructParams(kernel=H.KERNEL["centroid"], kmax=50, kmin=1, aca_eps=eps,
                            aca_eps_factor=H.baseline_params(aca_eps=eps)["aca_eps_factor"])
    I = C.POINTER(C.c_int)
    D = C.POINTER(C.c_double)
    d = C.c_void_p()
    L = H.hmv_lib()
    faces = np.ascontiguousarray(faces, np.int32)
    assert L.hmv_construct(len(nodes), nodes.ctypes.data_as(D), len(faces), faces.ctypes.data_as(I),
                           cent.ctypes.data_as(D), np.ascontiguousarray(area).ctypes.data_as(D),
                           lod.ctypes.data_as(I), len(blocks), C.addressof(rec), C.sizeof(H.LeafRec),
                           C.byref(cp), C.byref(d)) == 0, L.hmv_last_error()
    kt = np.zeros(len(blocks), np.int32)
    assert L.hmv_dleaves_info(d, None, kt.ctypes.data_as(I), None) == 0
    out = []
    for i, ((l0, ndl, t0, ndt), k) in enumerate(zip(blocks, kt)):
        buf = np.zeros((ndl + ndt) * max(int(k), 1))
        assert L.hmv_dleaves_download(d, i, buf.ctypes.data_as(D)) == 0
        V, U = buf[:ndt * k].reshape(k, ndt), buf[ndt * k:(ndt + ndl) * k].reshape(k, ndl)
        diff = cent[l0:l0 + ndl, None] - cent[None, t0:t0 + ndt]
        with np.errstate(divide="ignore"):
            A = area[None, t0:t0 + ndt] / (4 * np.pi * np.linalg.norm(diff, axis=2))
        out.append((U.T @ V, A, int(k)))
    L.hmv_dleaves_free(d)
    return out


@pytest.mark.parametrize("a,b", [(22, 300), (63, 65), (256, 257), (255, 1000), (2048, 257),
                                 (2049, 2048), (5120, 4097)])
def test_aca_workgroup_sizes(gpu, H, a, b):
    """ACA+ takes 64, 256 or 1024 threads by a block's longer side (up to 256,
    up to 2048, more).  Two far patches of a and b triangles, whose coupling is
    one block each way: ranks and factors of all leaves equal the host fill's
    bit for bit, as above."""
    n1, f1 = H.icosphere(4)
    n2, f2 = H.icosphere(4, 1.0, (30.0, 0.0, 0.0))
    nodes, faces = H.merge((n1, f1[:a]), (n2, f2[:b]))
    p = H.baseline_params(aca_eps=1e-6)
    host = H.HMatrix(nodes, faces, p)
    dev = H.DeviceHMatrix(nodes, faces, p)
    t = host.leaf_table()
    assert ((t[:, 0] == 1) & (t[:, 3] == a) & (t[:, 5] == b)).any()
    assert np.array_equal(dev.table, t)
    got = dev.download()
    for (kind, x, _), (_, y, _) in zip(_leaf_values(host, host.lod), _leaf_values(got, host.lod)):
        if kind == 1:
            assert np.array_equal(x, y)
    dev.free()


def test_aca_block_on_the_diagonal(gpu, H):
    """A block that holds diagonal entries evaluates them analytically (the
    kernel that knows no diagonal is for the other blocks): at full rank
    U V^T is the block, its diagonal the closed form of the self term."""
    nodes, faces = H.icosphere(1)
    n = 24
    (uv, A, k), = _construct_blocks(H, nodes, faces, [(0, n, 0, n)], 1e-15)
    tri = nodes[faces[:n]]
    cent = tri.mean(axis=1)
    self_term = np.zeros(n)
    for i in range(3):
        a, b = tri[:, i] - cent, tri[:, (i + 1) % 3] - cent
        e = (b - a) / np.linalg.norm(b - a, axis=1)[:, None]
        ta, tb = (a * e).sum(1), (b * e).sum(1)
        h = np.linalg.norm(a - ta[:, None] * e, axis=1)
        self_term += h * np.log((np.linalg.norm(b, axis=1) + tb) / (np.linalg.norm(a, axis=1) + ta))
    A[np.arange(n), np.arange(n)] = self_term / (4 * np.pi)
    print("rank", k, "error %.2e" % (np.linalg.norm(uv - A) / np.linalg.norm(A)), flush=True)
    assert np.linalg.norm(uv - A) / np.linalg.norm(A) < 1e-10


def test_ranks_at_the_stopping_test_itself(gpu, H):
    """A block's rank changes where one of its norms crosses its threshold.
    The two adjacent doubles aca_eps between which a rank of the host fill
    changes, for blocks of several sizes: the norm is within rounding of the
    threshold there, and the device takes the host's side on both."""
    mesh = H.icosphere(3)

    def table(eps):
        hm = H.HMatrix(*mesh, H.baseline_params(aca_eps=eps))
        t = hm.leaf_table()
        hm.close()
        return t

    above, below = table(1e-4), table(1e-5)
    change = np.nonzero(above[:, 1] != below[:, 1])[0]
    longest = np.maximum(above[change, 3], above[change, 5])
    for leaf in change[np.argsort(longest, kind="stable")][:: len(change) // 11]:
        hi, lo, k_hi = 1e-4, 1e-5, above[leaf, 1]
        while np.nextafter(lo, 1.0) < hi:
            mid = 0.5 * (lo + hi)
            if table(mid)[leaf, 1] == k_hi:
                hi = mid
            else:
                lo = mid
        for eps in (lo, hi):
            dev = H.DeviceHMatrix(*mesh, H.baseline_params(aca_eps=eps))
            assert np.array_equal(dev.table, table(eps)), (leaf, eps)
            dev.free()
