"""The split of wide phase-2 items (hmv::split_wide, host only) on the CPU: a
small program fills a plan's work list, splits it and prints the result."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "hacapk-magma_amd")

MAIN = r"""
#include <cstdio>
#include "hmv_plan.h"
// stdin: small items, instances (offsets), then "rows ncol0 ncol1 first_row"
int main() {
  hmv::Plan P;
  int n, ns;
  if (scanf("%d %d %d", &n, &P.nwork2_small, &ns) != 3) return 1;
  P.seg.resize(ns);
  for (int &s : P.seg) if (scanf("%d", &s) != 1) return 1;
  for (int i = 0; i < n; ++i) {
    HmvWork w{};
    if (scanf("%d %d %d %d", &w.rows, &w.ncol0, &w.ncol1, &w.out_base) != 4) return 1;
    w.rows_p = w.rows + (w.rows & 1);
    w.off0 = (int64_t)i << 40;
    w.off1 = ((int64_t)i << 40) + ((int64_t)1 << 36);
    w.dt0 = HMV_DT_F32;
    w.dt1 = HMV_DT_BF16;
    w.zseg_begin = (int)P.zseg.size();  // runs of 700 columns
    const int nc = w.ncol0 + w.ncol1;
    for (int c = 0; c < nc; c += 700)
      P.zseg.push_back(HmvZSeg{HMV_Z_X, nc - c < 700 ? nc - c : 700, 100000 + c, c});
    w.zseg_end = (int)P.zseg.size();
    P.work2.push_back(w);
  }
  hmv::WideSplit s;
  const int wide = hmv::split_wide(P, s);
  printf("%d %d %d\n", wide, s.nwork2_small, s.nyp);
  for (const HmvWork &w : s.work2) {
    printf("w %d %d %d %d %lld %lld", w.rows, w.ncol0, w.ncol1, w.out_base,
           (long long)w.off0, (long long)w.off1);
    for (int z = w.zseg_begin; z < w.zseg_end; ++z) {
      const HmvZSeg &g = z < (int)P.zseg.size() ? P.zseg[z] : s.zseg[z - P.zseg.size()];
      printf(" %d %d %d", g.col, g.ncols, g.src);
    }
    printf("\n");
  }
  for (const HmvYFin &f : s.yfin)
    printf("f %d %d %d %d %d\n", f.row, f.rows, f.base, f.np, f.inst);
}
"""


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    d = tmp_path_factory.mktemp("wide")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"), "-I",
                    os.path.join(ROOT, "include"), str(d / "main.cpp"),
                    os.path.join(PKG, "csrc", "hmv_plan.cpp"), "-pthread", "-o", str(d / "main")],
                   check=True, timeout=300)

    def run(items, small=0, seg=(0, 10 ** 6)):
        text = "%d %d %d %s\n" % (len(items), small, len(seg), " ".join(map(str, seg)))
        text += "\n".join(" ".join(map(str, it)) for it in items)
        p = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True,
                           check=True, timeout=60)
        lines = [ln.split() for ln in p.stdout.splitlines()]
        head = list(map(int, lines[0]))
        return (head, [list(map(int, t[1:])) for t in lines if t[0] == "w"],
                [list(map(int, t[1:])) for t in lines if t[0] == "f"])

    return run


def _check(items, seg, head, work, fin):
    """Every item whole, or in pieces that hold its columns, runs and offsets
    once each, with rows of their own among the partial rows."""
    taken = np.zeros(head[2], int)
    by_base = {f[2]: f for f in fin}
    whole = [w for w in work if w[3] >= 0]
    pieces = {}
    for w in work:
        if w[3] < 0:
            base = -1 - w[3]
            f = by_base[max(b for b in by_base if b <= base)]
            pieces.setdefault(f[0], []).append(((base - f[2]) // f[1], w))
            taken[base:base + w[0]] += 1
    assert np.all(taken == 1)
    assert len(whole) + len(pieces) == len(items) and len(fin) == len(pieces)
    for i, (rows, n0, n1, row) in enumerate(items):
        if row not in pieces:
            assert any(w[:4] == [rows, n0, n1, row] for w in whole)
            continue
        f = next(f for f in fin if f[0] == row)
        assert f[1] == rows and f[3] == len(pieces[row]) >= 2
        assert seg[f[4]] <= row < seg[f[4] + 1]
        col, rows_p = 0, rows + rows % 2
        for q, (at, w) in enumerate(sorted(pieces[row])):
            assert at == q and w[0] == rows and 0 < w[1] + w[2] <= 1024
            c0, c1 = min(col, n0), max(0, col - n0)
            assert w[4] == (i << 40) + c0 * rows_p * 4
            assert w[5] == (i << 40) + (1 << 36) + c1 * rows_p * 2
            assert w[1] == min(col + w[1] + w[2], n0) - c0
            runs = np.array(w[6:]).reshape(-1, 3)
            covered = np.concatenate([np.arange(s, s + n) for _, n, s in runs])
            assert np.array_equal(covered, 100000 + col + np.arange(w[1] + w[2]))
            assert np.array_equal(runs[:, 0], np.concatenate([[0], np.cumsum(runs[:, 1])[:-1]]))
            col += w[1] + w[2]
        assert col == n0 + n1


def test_pieces_cover_their_items(split):
    items = [(40, 3071, 0, 0), (40, 3072, 0, 40), (33, 100, 3000, 80), (256, 3500, 0, 200),
             (7, 20001, 13, 600), (50, 800, 0, 700), (64, 0, 5000, 800)]
    seg = (0, 150, 600, 1000)
    head, work, fin = split(items, small=3, seg=seg)
    assert head[0] == 1 and len(fin) == 5
    _check(items, seg, head, work, fin)
    # the first head[1] of the list are the pieces and items of the first three
    assert sum(w[0] in (40, 33) for w in work[:head[1]]) == head[1]
    assert sum(w[0] in (40, 33) for w in work) == head[1]
    head, work, fin = split(items[:1])
    assert head[0] == 0 and not work and not fin


def test_partial_rows_have_a_limit(split):
    """More wide rows than HMV_PARTIAL_ROWS (65,536): the widest in pieces as
    far as they go, the others whole."""
    items = [(250, 3072 + (i % 3) * 1024, 0, 250 * i) for i in range(100)]
    seg = (0, 25000)
    head, work, fin = split(items, seg=seg)
    _check(items, seg, head, work, fin)
    # 33 items of 5 pieces (41,250 rows), then 24 of 4 (24,000): 286 rows are left
    assert head[2] == 65250
    cut = [items[f[0] // 250][1] for f in fin]
    assert sorted(cut) == [4096] * 24 + [5120] * 33
