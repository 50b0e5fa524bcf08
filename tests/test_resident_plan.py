"""Plans of the resident solves on the CPU: every neighbour of every node is
found where the plan says (own position or halo entry), the halo lists name
published nodes, and the pieces cover each aggregate's chunks."""

import numpy as np
import pytest
import torch
from scipy.spatial import Delaunay

import easyfea_amd as ea
from easyfea_amd import resident as R
from easyfea_amd._lib import EfeaError
from easyfea_amd.assembly_map import build_csr_map
from easyfea_amd.coarse import aggregate
from easyfea_amd.mesh import tetra4_box


def _with_orphans(mesh, at):
    """The mesh with nodes of no element inserted before the nodes ``at``
    (Nn: after the last one)."""
    at = np.asarray(at)
    new = np.arange(mesh.Nn) + np.searchsorted(at, np.arange(mesh.Nn), side="right")
    coord = np.insert(mesh.coord, at, mesh.coord[np.minimum(at, mesh.Nn - 1)] + 0.01, axis=0)
    return ea.Mesh({t: new[g.connect] for t, g in mesh.dict_groupElem.items()}, coord)


def irregular(n, dim, seed=0):
    """Delaunay triangles or tetrahedra of an (n + 1)^dim grid whose inner
    points are moved by up to 0.45 of a cell; flat ones left out."""
    g = np.stack(np.meshgrid(*[np.arange(n + 1.0)] * dim, indexing="ij"), -1).reshape(-1, dim)
    move = np.random.default_rng(seed).uniform(-0.45, 0.45, g.shape)
    g += np.where((g > 0) & (g < n), move, 0.0)
    con = Delaunay(g).simplices
    con = con[np.abs(np.linalg.det(g[con[:, 1:]] - g[con[:, :1]])) > 1e-3]
    coord = np.zeros((len(g), 3))
    coord[:, :dim] = g / n
    return ea.Mesh({"TRI3" if dim == 2 else "TETRA4": con}, coord)


MESHES = {
    "irregular 2D": (lambda: irregular(30, 2, 2), 2),
    "irregular 3D": (lambda: irregular(8, 3), 3),
    # empty rows first, in the middle and last
    "orphans quad 20": (lambda: _with_orphans(ea.quad4_rectangle(1.0, 1.0, 20, 20), [0, 200, 200, 441]), 2),
    "orphan tetra 5": (lambda: _with_orphans(tetra4_box(1.0, 1.0, 1.0, 5, 5, 5), [216]), 3),
    "one cell": (lambda: ea.quad4_rectangle(1.0, 1.0, 1, 1), 2),
    "quad 33x17": (lambda: ea.quad4_rectangle(2.0, 1.0, 33, 17), 2),
    "notched 40": (lambda: ea.tri3_notched_square(40), 2),
    "hexa 9x8x11": (lambda: ea.hexa8_box(1.0, 1.0, 1.0, 9, 8, 11), 3),
    "tetra 7": (lambda: tetra4_box(1.0, 1.0, 1.0, 7, 7, 7), 3),
}


def _plan(name, dof_n, target, blocks):
    mesh = MESHES[name][0]()
    m = build_csr_map(mesh.connect, mesh.Nn, dof_n)
    ag = None if target is None else aggregate(mesh.coord, m.node_ptr, m.node_cols, target)
    lay = R.layout(mesh.coord, mesh.Nn, dof_n, m.max_neighbours, blocks, ag)
    return mesh, m, ag, lay


@pytest.mark.parametrize("name,scalar,target,blocks", [
    (n, s, t, b) for n in MESHES for s, t, b in [(True, None, 256), (False, None, 256), (False, 40, 256),
                                                 (False, 40, 9)]])
def test_plan_covers_the_matrix(name, scalar, target, blocks):
    dof_n = 1 if scalar else MESHES[name][1]
    mesh, m, ag, lay = _plan(name, dof_n, target, blocks)
    if lay is None:
        assert blocks == 9  # more chunks than nine blocks hold
        return
    lanes, slots, passes, rows, chunk_agg = lay
    nblk, nloc = rows.shape
    assert nblk <= blocks and nloc == 512 // lanes * passes and lanes * slots >= m.max_neighbours
    assert np.array_equal(np.sort(rows[rows >= 0]), np.arange(mesh.Nn))
    nb = R.neighbours(torch.from_numpy(rows), torch.from_numpy(m.node_ptr), torch.from_numpy(m.node_cols), lanes,
                      slots, passes)
    hp, hx, pub = (nb[k].numpy() for k in ("halo_ptr", "halo_ex", "pub"))
    assert hp[0] == 0 and hp[-1] == hx.size and np.diff(hp).max() == nb["max_halo"]
    owner = np.full(nb["nex"], -1)  # exchange number -> node
    owner[pub[pub >= 0]] = rows.ravel()[pub >= 0]
    assert (owner >= 0).all() and (pub >= 0).sum() == nb["nex"]
    kept = slots - 1 if scalar else slots  # a scalar row's own node has no entry
    lidx = nb["lidx"].numpy().view(np.uint16).reshape(nblk, passes, kept, 512)
    pp, ppos, self_k = (nb[k].numpy() for k in ("pub_ptr", "pub_pos", "self"))
    assert pp[0] == 0 and pp[-1] == nb["nex"]
    assert lidx.max() < nloc + max(nb["max_halo"], 1)
    per = 64 // lanes
    seen = 0
    for b in range(nblk):
        assert np.array_equal(pub[b * nloc + ppos[pp[b]:pp[b + 1]]], np.arange(pp[b], pp[b + 1]))
        local = np.concatenate([rows[b], owner[hx[hp[b]:hp[b + 1]]]])
        for p in np.nonzero(rows[b] >= 0)[0]:
            n, chunk = rows[b, p], p // per
            cols = m.node_cols[m.node_ptr[n]:m.node_ptr[n + 1]]
            if scalar and cols.size:
                assert cols[self_k[b * nloc + p]] == n
                cols = np.delete(cols, self_k[b * nloc + p])
            k = np.arange(cols.size)
            t = (chunk % 8) * 64 + (p % per) * lanes + k % lanes
            assert np.array_equal(local[lidx[b, chunk // 8, k // lanes, t]], cols)
            seen += 1
    assert seen == mesh.Nn
    if ag is not None:
        pc = R.pieces(chunk_agg)
        for b in range(nblk):
            ch = rows[b].reshape(-1, per)
            for j in range(pc["piece_ptr"][b], pc["piece_ptr"][b + 1]):
                c0, c1 = pc["piece_chunk"][2 * j:2 * j + 2]
                assert c0 < c1 and (chunk_agg[b, c0:c1] == pc["piece_agg"][j]).all()
                assert (pc["chunk_piece"].reshape(nblk, -1)[b, c0:c1] == j - pc["piece_ptr"][b]).all()
                nodes = ch[c0:c1][ch[c0:c1] >= 0]
                assert (ag.agg[nodes] == pc["piece_agg"][j]).all()
        assert np.array_equal(np.unique(pc["piece_agg"]), np.arange(ag.nagg))
        nm = 3 if MESHES[name][1] == 2 else 6
        _check_collection(R.collection(nm, ag.nagg, pc), nblk, nm, pc)


def _check_collection(table, nblk, nm, pc):
    """Every component gathers its aggregate's pieces in block order."""
    line = -(-(3 + nm * pc["max_pieces"]) // 8) * 8
    got, run = {}, []
    for t in range(R.COLLECTORS):
        for e in table[:, t]:
            if e == -1:
                assert not run
                continue
            run.append(int(e) & 0xffff)
            if e < -1:
                got[(int(e) >> 16) & 0x7fff] = run
                run = []
    want = {}
    for k in range(nblk):
        for i, j in enumerate(range(pc["piece_ptr"][k], pc["piece_ptr"][k + 1])):
            for m in range(nm):
                want.setdefault(pc["piece_agg"][j] * nm + m, []).append(k * line + 3 + i * nm + m)
    assert got == want


@pytest.mark.parametrize("n,parts", [(1, 1), (7, 3), (5000, 17), (300_000, 256)])  # the last one by several threads
def test_bisection_parts(n, parts):
    rng = np.random.default_rng(n)
    coord = np.zeros((n, 3))
    coord[:, :2] = rng.integers(0, 600, (n, 2))  # many equal coordinates
    coord[rng.integers(0, n, 3), 2] = [0.0, np.inf, np.nan]
    out = R.bisect(coord, parts)
    assert len(out) == parts and np.array_equal(np.sort(np.concatenate(out)), np.arange(n))
    assert all((np.diff(p) > 0).all() and p.size <= -(-n // parts) for p in out)
    again = R.bisect(coord, parts)
    assert all(np.array_equal(a, b) for a, b in zip(out, again))
    plane = R.bisect(np.asfortranarray(coord[:, :2]), parts)
    assert sum(p.size for p in plane) == n


def test_neighbours_refuses_rows_that_do_not_fit():
    mesh, m, _, (lanes, slots, passes, rows, _) = _plan("quad 33x17", 1, None, 256)
    graph = torch.from_numpy(m.node_ptr), torch.from_numpy(m.node_cols)
    for bad in (np.where(rows == 5, -1, rows), np.where(rows == 5, mesh.Nn, rows)):  # a node without a place, none
        with pytest.raises(EfeaError, match="position"):
            R.neighbours(torch.from_numpy(bad), *graph, lanes, slots, passes)
    with pytest.raises(EfeaError, match="slots"):
        R.neighbours(torch.from_numpy(rows), *graph, lanes, slots - 2, passes)
    with pytest.raises(EfeaError, match="lanes"):
        R.neighbours(torch.from_numpy(rows), *graph, 3, slots, passes)


def test_layout_refuses_what_no_variant_holds():
    assert R.shape(2, 17, 1) is None and R.shape(3, 29, 1) is None and R.shape(1, 29, 1) is None
    coord = np.random.default_rng(0).uniform(size=(3000, 3))
    assert R.layout(coord, 3000, 3, 27, 23, None) is None  # 128 nodes a block
    lanes, slots, passes, rows, _ = R.layout(coord, 3000, 3, 27, 24, None)
    assert (lanes, slots, passes) == (4, 7, 1) and rows.shape == (24, 128)
