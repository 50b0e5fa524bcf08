"""Assembly by rows (``efea_elastic_assemble``) against the oracle's element
matrices summed on the host, over every element type, sizes that leave a part of
the last block's nodes empty, shuffled connectivity, and the meshes it leaves to
the element-matrix path.

Bar per entry: 1e-14 (the bar of the element matrices themselves) of the sum,
over the elements of the entry, of each one's largest entry."""

import numpy as np
import pytest
import scipy.sparse as sp

import easyfea_amd as ea
from easyfea_amd import Models, Simulations, _lib
from easyfea_amd.assembly_map import build_csr_map
from easyfea_amd.device import DeviceMesh
from easyfea_amd.mesh import tetra4_box, tetra10_from_tetra4
from oracle import efea_oracle as O

MESHES = {
    "TRI3": lambda k: ea.tri3_rectangle(3.0, 2.0, 6 + k, 5),
    "QUAD4": lambda k: ea.quad4_rectangle(3.0, 2.0, 6 + k, 5),
    "HEXA8": lambda k: ea.hexa8_box(1.0, 2.0, 1.5, 3 + k, 3, 5),
    "TETRA4": lambda k: tetra4_box(1.0, 2.0, 1.5, 2 + k, 2, 4),
    "TETRA10": lambda k: tetra10_from_tetra4(tetra4_box(1.0, 2.0, 1.5, 2 + k, 2, 3)),
}


def _mesh(et, k, seed=0):
    """Distorted, elements in random order."""
    mesh = MESHES[et](k)
    rng = np.random.default_rng(seed)
    c = mesh.coord.copy()
    h = (c.max(0) - c.min(0))[:mesh.dim].min() / 12
    c[:, :mesh.dim] += 0.2 * h * (rng.random((mesh.Nn, mesh.dim)) - 0.5)
    (t, g), = [(t, g) for t, g in mesh.dict_groupElem.items() if g.dim == mesh.dim]
    return ea.Mesh({t: g.connect[rng.permutation(g.Ne)]}, c)


def _reference(mesh, et, C, thickness):
    Ke = O.K_elastic(O.Geometry(et, mesh.connect, mesh.coord, "rigi", mesh.dim), C) * thickness
    con, dim = mesh.connect, mesh.dim
    dofs = (con[:, :, None] * dim + np.arange(dim)).reshape(len(con), -1)
    n = dofs.shape[1]
    ij = np.repeat(dofs, n, axis=1).ravel(), np.tile(dofs, (1, n)).ravel()
    size = np.repeat(np.abs(Ke).max(axis=(1, 2)), n * n)
    shape = (mesh.Nn * dim,) * 2
    return [sp.coo_matrix((v, ij), shape=shape).toarray() for v in (Ke.ravel(), size)]


def _assembled(mesh, law):
    simu = Simulations.Elastic(mesh, law)
    A = simu.Assembly()
    assert simu.dev.row_incidence(mesh.dim) is not None
    return A.to_scipy().toarray()


@pytest.mark.gpu
@pytest.mark.parametrize("k", [0, 1, 2])
@pytest.mark.parametrize("et,planeStress,het", [
    ("TRI3", True, True), ("TRI3", False, False), ("QUAD4", True, False), ("QUAD4", False, True),
    ("HEXA8", False, True), ("HEXA8", False, False), ("TETRA4", False, True), ("TETRA10", False, True),
])
def test_isotropic_rows(et, planeStress, het, k):
    mesh = _mesh(et, k, seed=k)
    dim = mesh.dim
    E = 210000.0 * np.exp(0.2 * np.random.default_rng(1).standard_normal(mesh.Ne)) if het else 210000.0
    thickness = 13.0 if dim == 2 else 1.0
    law = Models.Elastic.Isotropic(dim, E, 0.3, planeStress=planeStress, thickness=thickness)
    ref, size = _reference(mesh, et, O.C_isotropic(E, 0.3, dim, planeStress), thickness)
    K = _assembled(mesh, law)
    worst = np.max(np.abs(K - ref) / np.where(size > 0, size, 1.0))
    print(f"{et} {worst:.1e}")
    assert worst < 1e-14


@pytest.mark.gpu
@pytest.mark.parametrize("per_element", [False, True])
@pytest.mark.parametrize("et", ["HEXA8", "TETRA10"])
def test_general_rows(et, per_element):
    mesh = _mesh(et, 1, seed=5)
    Q = np.random.default_rng(2).standard_normal((mesh.Ne if per_element else 1, 6, 6))
    C = 1e4 * (Q @ np.swapaxes(Q, 1, 2) + 6 * np.eye(6))
    law = Models.Elastic.Anisotropic(3, C if per_element else C[0], False)
    ref, size = _reference(mesh, et, law.C, 1.0)
    worst = np.max(np.abs(_assembled(mesh, law) - ref) / np.where(size > 0, size, 1.0))
    assert worst < 1e-14


def _fan(n):
    """n triangles around one node."""
    t = 2 * np.pi * np.arange(n) / n
    coord = np.zeros((n + 1, 3))
    coord[1:, 0], coord[1:, 1] = np.cos(t), np.sin(t)
    i = np.arange(n)
    return ea.Mesh({"TRI3": np.stack([0 * i, 1 + i, 1 + (i + 1) % n], axis=1)}, coord)


@pytest.mark.gpu
def test_longest_rows_and_the_ones_beyond():
    most = _lib.load().efea_assemble_max_neighbours(_lib.ELEM_CODE["TRI3"])
    law = Models.Elastic.Isotropic(2, 210000.0, 0.3)
    for n, fits in [(most - 1, True), (most, False)]:  # the hub's row holds the hub itself as well
        mesh = _fan(n)
        simu = Simulations.Elastic(mesh, law)
        K = simu.Assembly().to_scipy().toarray()
        assert (simu.dev.row_incidence(2) is not None) is fits
        ref, size = _reference(mesh, "TRI3", O.C_isotropic(210000.0, 0.3, 2, law.planeStress), law.thickness)
        assert np.max(np.abs(K - ref) / np.where(size > 0, size, 1.0)) < 1e-14


@pytest.mark.gpu
@pytest.mark.parametrize("dof_n", [1, 2, 3])
@pytest.mark.parametrize("et", list(MESHES))
def test_row_incidence_lists_each_pair_once(et, dof_n):
    mesh = _mesh(et, 1)
    m = build_csr_map(mesh.connect, mesh.Nn, 1)
    inc_ptr, inc, pos = (a.cpu().numpy() for a in DeviceMesh(mesh).row_incidence(dof_n))
    assert inc_ptr[-1] == mesh.connect.size == len(inc) == len(pos)
    for n in range(mesh.Nn):
        rows = slice(inc_ptr[n], inc_ptr[n + 1])
        e = inc[rows] >> 4
        assert np.all(np.diff(e) > 0)
        assert np.all(mesh.connect[e, inc[rows] & 15] == n)
        row = m.node_cols[m.node_ptr[n]:m.node_ptr[n + 1]]
        assert np.array_equal(row[pos[rows]], mesh.connect[e])


@pytest.mark.parametrize("dof_n", [1, 2])
def test_the_map_tells_a_repeated_node(dof_n):
    con = ea.quad4_rectangle(3.0, 2.0, 4, 3).connect
    assert not build_csr_map(con, 21, dof_n).repeated  # (and a node of no element)
    for k in range(3):
        twice = con.copy()
        twice[7, 3] = twice[7, k]
        assert build_csr_map(twice, 21, dof_n).repeated


@pytest.mark.gpu
def test_a_repeated_node_keeps_element_matrices():
    """A QUAD4 mesh whose last element is collapsed to a triangle."""
    mesh = ea.quad4_rectangle(3.0, 2.0, 4, 3)
    con = mesh.connect.copy()
    con[-1, 3] = con[-1, 2]
    mesh = ea.Mesh({"QUAD4": con}, mesh.coord)
    law = Models.Elastic.Isotropic(2, 210000.0, 0.3)
    simu = Simulations.Elastic(mesh, law)
    K = simu.Assembly().to_scipy().toarray()
    assert simu.dev.row_incidence(2) is None
    ref, size = _reference(mesh, "QUAD4", O.C_isotropic(210000.0, 0.3, 2, law.planeStress), law.thickness)
    assert np.max(np.abs(K - ref) / np.where(size > 0, size, 1.0)) < 1e-14
