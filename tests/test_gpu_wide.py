"""Phase-2 items of 3,072 columns and more run as pieces whose partial rows a
last launch sums: products of leaf sets with such items, at and around that
width, against the oracle (FP64 within 1e-12, narrow storage within the
bounds of the other apply tests)."""
import numpy as np
import pytest
from synthetic_leaves import LeafSet

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 1e-5, "bf16": 2e-2, "bf16_all": 2e-2}


def _leaves(H, nd=9100, seed=3):
    lv = [("dense", 0, 1, 0, 3071, 0), ("dense", 1, 2, 10, 3072, 0), ("dense", 3, 17, 5, 3073, 0),
          ("dense", 20, 13, 0, 9001, 0), ("lowrank", 20, 13, 40, 3000, 7),
          # one wide item of dense and low-rank columns (two parts where they
          # are stored apart) under row clusters of several sizes
          ("dense", 40, 30, 100, 3500, 0), ("lowrank", 36, 64, 0, 4000, 9),
          ("lowrank", 40, 30, 5000, 100, 40), ("lowrank", 33, 200, 3000, 6000, 12)]
    # more input runs than the run table: 100 dense leaves of 41 columns
    lv += [("dense", 300, 20, 60 * j, 41, 0) for j in range(100)]
    # the most rows of one item, wide; ordinary items
    lv += [("dense", 400, 256, 0, 3600, 0), ("dense", 700, 40, 50, 600, 0),
           ("lowrank", 680, 300, 2000, 500, 6)]
    return LeafSet(H, nd, lv, seed)


@pytest.fixture(scope="module")
def wide(gpu):
    return _leaves(gpu)


def _err(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("prec", ["f64", "f32", "bf16", "bf16_all"])
def test_wide_items(gpu, O, wide, tmp_path, prec):
    a = gpu.Arena(wide, prec)
    x = gpu.uniform(1, wide.nd)
    ref = O.adot_body_lfmtx(wide, x)
    y = a.matvec(x)
    assert _err(y, ref) <= TOL[prec]
    dx, dy = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer.from_array(2 * x)
    a.apply(dx.ptr, dy.ptr, 1.0)
    assert _err(dy.download() - 2 * x, ref) <= TOL[prec]
    assert np.array_equal(a.matvec(x), y)
    for k in (1, 3, 8, 19, 33, 128):
        X = np.stack([gpu.uniform(10 + j, wide.nd) for j in range(k)], axis=1)
        Y = a.matmat(X)
        for j in sorted({0, k // 2, k - 1}):
            assert _err(Y[:, j], O.adot_body_lfmtx(wide, X[:, j])) <= TOL[prec], (k, j)
    # the file holds the items whole, and an arena from it runs the same
    a.save(tmp_path / "a.hmv")
    b = gpu.Arena.load(tmp_path / "a.hmv")
    assert np.array_equal(b.matvec(x), y)
    b.save(tmp_path / "b.hmv")
    assert (tmp_path / "a.hmv").read_bytes() == (tmp_path / "b.hmv").read_bytes()
    a.free()
    b.free()


def test_wide_items_of_instances(gpu, O, wide):
    other = _leaves(gpu, nd=9050, seed=5)
    m = gpu.MultiArena([wide, other], "f64")
    x = gpu.uniform(2, m.nd)
    y = m.matvec(x)
    for hm, lo, hi in ((wide, 0, wide.nd), (other, wide.nd, m.nd)):
        assert _err(y[lo:hi], O.adot_body_lfmtx(hm, x[lo:hi])) <= 1e-12
    m.free()


def test_partial_rows_are_bounded(gpu, O):
    """More wide rows than the partial buffer holds: the widest run in pieces,
    the others whole."""
    nd = 8000
    lv = [("dense", 64 * i, 64, 0, 2048 + 48 * i, 0) for i in range(120)]
    hm = LeafSet(gpu, nd, lv, 9)
    assert sum(nr * -(-nc // 1024) for _, _, nr, _, nc, _ in lv if nc >= 3072) < 65536
    tall = LeafSet(gpu, 80000, [("dense", 250 * i, 250, 0, 3072, 0) for i in range(150)], 10)
    assert 150 * 250 * 3 > 65536
    for s in (hm, tall):
        a = gpu.Arena(s, "f64")
        x = gpu.uniform(4, s.nd)
        assert _err(a.matvec(x), O.adot_body_lfmtx(s, x)) <= 1e-12
        a.free()


@pytest.fixture(scope="module")
def tall(gpu):
    """75,000 rows of wide items in three pieces each: more partial rows than
    an arena may have."""
    return LeafSet(gpu, 80000, [("dense", 250 * i, 250, 0, 3072, 0) for i in range(100)], 10)


@pytest.mark.parametrize("name,prec,k", [
    ("wide", "f64", 1), ("wide", "f64", 8), ("wide", "f64", 19), ("wide", "f64", 128),
    ("wide", "bf16", 33), ("tall", "f64", 3), ("tall", "f64", 128)])
def test_wide_items_without_allocation(gpu, request, name, prec, k):
    """hmv_apply_block_static on wide items: the partial rows are the arena's
    own; the same kernels and sums as hmv_apply_block, bit for bit, also with
    the most partial rows."""
    hm = request.getfixturevalue(name)
    a = gpu.Arena(hm, prec)
    X = np.stack([gpu.uniform(20 + j, hm.nd) for j in range(k)], axis=1)
    want = a.matmat(X)
    dx = gpu.DeviceBuffer.from_array(X.reshape(-1))
    dy = gpu.DeviceBuffer.from_array(np.full(X.size, np.nan))
    gpu._check(gpu.hmv_lib().hmv_apply_block_static(a.handle, k, dx.ptr, dy.ptr, 0.0, None),
               "hmv_apply_block_static")
    gpu.hmv_lib().hmv_device_synchronize()
    assert np.array_equal(dy.download().reshape(hm.nd, k), want)
    dx.free()
    dy.free()
    a.free()


class _Solvable(LeafSet):
    """A well-conditioned matrix with wide items: 40 full rows among diagonal
    blocks, and a low-rank block."""

    def __init__(self, H, nd, seed):
        at = [0, 700, nd - 40]  # first of the full rows: 40 at one of these
        top = at[seed % 3]
        lv = [("dense", top, 40, 0, nd, 0)]
        for lo, hi in ((0, top), (top + 40, nd)):
            lv += [("dense", r, min(60, hi - r), r, min(60, hi - r), 0) for r in range(lo, hi, 60)]
        lv.append(("lowrank", 100, 300, nd - 900, 400, 3))
        super().__init__(H, nd, lv, seed)
        self.A = np.zeros((nd, nd))
        for (kind, r0, nr, c0, nc, k), buf in zip(lv, self._bufs):
            if kind == "dense":
                block = buf.reshape(nr, nc)
                block *= 0.05
                i = np.arange(nr)
                block[i, i + r0 - c0] += 3.0 + 0.01 * i
                self.A[r0:r0 + nr, c0:c0 + nc] += block
            else:
                buf *= 0.1
                v, u = buf[:nc * k].reshape(k, nc), buf[nc * k:].reshape(k, nr)
                self.A[r0:r0 + nr, c0:c0 + nc] += u.T @ v


@pytest.mark.parametrize("early", [0, 1, 2])
def test_instances_with_wide_items_stop_on_their_own(gpu, O, early):
    """Three instances with wide items, one of which starts at its solution:
    its pieces and their sums are skipped from then on, the others' are not
    (each instance's solution is that of its dense matrix)."""
    hms = [_Solvable(gpu, nd, s) for s, nd in enumerate((3200, 3411, 3100))]
    m64, low = gpu.MultiArena(hms, "f64"), gpu.MultiArena(hms, "f32")
    off = np.cumsum([0] + [hm.nd for hm in hms])
    b = gpu.uniform(30 + early, m64.nd)
    want = np.concatenate([np.linalg.solve(hm.A, b[lo:hi])
                           for hm, lo, hi in zip(hms, off, off[1:])])
    assert _err(O.adot_body_lfmtx(hms[early], want[off[early]:off[early + 1]]),
                b[off[early]:off[early + 1]]) < 1e-13
    u0 = np.zeros(m64.nd)
    u0[off[early]:off[early + 1]] = want[off[early]:off[early + 1]]
    for name, (u, inst, *_) in (
            ("bicgstab", m64.bicgstab_multi(b, u0, eps=1e-10)),
            ("bicgstab_ir", gpu.multi_bicgstab_ir(m64, low, b, u0, eps=1e-10)),
            ("gcr_ir", gpu.multi_gcr_ir(m64, low, b, u0, eps=1e-10))):
        steps = [i["nstp"] for i in inst]
        print(name, "steps", steps, flush=True)
        assert [s == 0 for s in steps] == [i == early for i in range(3)]
        for i, (lo, hi) in enumerate(zip(off, off[1:])):
            assert inst[i]["status_name"] == "converged"
            assert _err(u[lo:hi], want[lo:hi]) < 1e-8, (name, i)
    m64.free()
    low.free()
