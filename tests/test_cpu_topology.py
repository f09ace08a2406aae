"""The native host part of scene compilation (wc_topology.cpp) against plain
restatements: edge candidates with their public ids (reference
scene/resources.py:79-148, 286-404) on meshes with shared, boundary,
non-manifold, welded-apart and degenerate edges, and the hulls of coplanar
groups."""

from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from witwin.channel import workloads
from witwin.channel.scene import compiler


def _edge_table(vertices, faces, face_group, face_structure, base):
    """(vertex ids, public id) of every candidate edge, dictionary by dictionary."""
    q = np.rint(vertices.astype(np.float64) / compiler.EDGE_WELD_QUANTIZATION).astype(np.int64)
    ids, cursor = {}, 0
    for s in range(len(base)):
        pairs = sorted({(min(a, b), max(a, b)) for f in faces[face_structure == s] - base[s]
                        for a, b in ((f[0], f[1]), (f[1], f[2]), (f[2], f[0]))})
        ids.update({(s, *p): cursor + r for r, p in enumerate(pairs)})
        cursor += len(pairs)
    table = {}
    for f, idx in enumerate(faces):
        for k in range(3):
            i = [int(idx[(k + j) % 3]) for j in range(3)]
            a, b = tuple(q[i[0]]), tuple(q[i[1]])
            la, lb = (x - base[face_structure[f]] for x in i[:2])
            table.setdefault((min(a, b), max(a, b)), []).append(
                (f, *i, ids[(face_structure[f], min(la, lb), max(la, lb))]))
    out = []
    for entries in table.values():
        if len(entries) == 1:
            out.append((*entries[0][1:4], -1, entries[0][4]))
        elif len(entries) == 2 and face_group[entries[0][0]] != face_group[entries[1][0]]:
            out.append((*entries[0][1:4], entries[1][3], min(entries[0][4], entries[1][4])))
    return sorted(out, key=lambda e: e[4])


def _random_mesh(seed):
    rng = np.random.default_rng(seed)
    corners = rng.uniform(-5.0, 5.0, (14, 3)).astype(np.float32)
    vertices = np.concatenate([corners, corners[:6] + np.float32(2e-6), corners[6:9] + np.float32(1e-3)])
    faces = rng.integers(0, 12, (24, 3))
    faces = faces[(faces[:, 0] != faces[:, 1]) & (faces[:, 1] != faces[:, 2]) & (faces[:, 2] != faces[:, 0])]
    # a second structure on the welded copies (vertices 14 ..)
    more = rng.integers(0, 9, (12, 3))
    more = more[(more[:, 0] != more[:, 1]) & (more[:, 1] != more[:, 2]) & (more[:, 2] != more[:, 0])]
    structure = np.concatenate([np.zeros(len(faces), np.int64), np.ones(len(more), np.int64)])
    return vertices, np.concatenate([faces, more + 14]).astype(np.int32), structure, np.array([0, 14])


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
def test_edge_candidates_match_restatement(seed):
    vertices, faces, structure, base = _random_mesh(seed)
    group = np.arange(len(faces), dtype=np.int32) // 2
    edges, ev, public = compiler.build_edge_table(vertices, faces, group, np.zeros(len(faces), np.int32),
                                                  face_structure=structure, structure_vertex_base=base,
                                                  return_ids=True)
    ref = _edge_table(vertices, faces, group, structure, base)
    g = compiler.edge_geometry(vertices, np.array([e[:4] for e in ref]).reshape(-1, 4))
    keep = (g["length"] >= 1e-9) & ~(g["wedge"] & ((np.abs(g["alpha"] - np.pi) < compiler.COPLANAR_ANGLE_TOLERANCE)
                                                   | (g["alpha"] < 1e-6)))
    ref = [e for e, k in zip(ref, keep) if k]
    assert len(ref) > 0 and [tuple(map(int, e)) for e in ev] == [tuple(map(int, e[:4])) for e in ref]
    assert public.tolist() == [int(e[4]) for e in ref] and edges.shape[0] == len(ref)


def test_edge_candidates_refuse_an_unknown_structure():
    vertices, faces, structure, base = _random_mesh(1)
    with pytest.raises(RuntimeError, match="structure"):
        compiler.build_edge_table(vertices, faces, np.arange(len(faces), dtype=np.int32),
                                  np.zeros(len(faces), np.int32), face_structure=structure + 1,
                                  structure_vertex_base=base)


@pytest.mark.parametrize("vertex", [23, 2 ** 32, -24])
def test_faces_outside_the_vertices_are_refused(vertex):
    vertices, faces, _, _ = _random_mesh(1)
    assert len(vertices) == 23
    faces = faces.astype(np.int64)
    faces[-1, 2] = vertex
    n = len(faces)
    with pytest.raises(IndexError):
        compiler.build_edge_table(vertices, faces, np.arange(n), np.zeros(n, np.int32))
    with pytest.raises(IndexError):
        compiler.group_hulls(vertices, faces, np.arange(n + 1), np.arange(n), np.tile([0.0, 0.0, 1.0, 0.0], (n, 1)))


def test_short_tables_are_refused():
    vertices, faces, structure, base = _random_mesh(1)
    n = len(faces)
    group, material = np.arange(n), np.zeros(n, np.int32)
    for tables in ((group[:-1], material, structure), (group, material[:-1], structure),
                   (group, material, structure[:-1])):
        with pytest.raises(IndexError):
            compiler.build_edge_table(vertices, faces, tables[0], tables[1], face_structure=tables[2],
                                      structure_vertex_base=base)
    plane = np.tile([0.0, 0.0, 1.0, 0.0], (n, 1))
    for offset, listed in ((np.arange(n), np.arange(n)), (np.arange(n + 1), np.arange(1, n + 1))):
        with pytest.raises(IndexError):
            compiler.group_hulls(vertices, faces, offset, listed, plane)
    with pytest.raises(RuntimeError, match="group"):
        compiler.group_hulls(vertices, faces, np.arange(n + 1), np.arange(n - 1), plane)


@pytest.mark.parametrize("first,loaded", [("", ["False", "True"]), ("_native.load();", ["True", "False"])])
def test_compiling_a_scene_loads_one_library(first, loaded):
    """In a process of its own: the host library, since libwcmi.so opened before
    the GPU runtime slows every later allocation and launch; with libwcmi.so
    open, none after it, for the same reason."""
    code = ("import torch; from witwin.channel import _native, workloads; from witwin.channel.scene import compiler;"
            f"{first}"
            "compiler.compile(workloads.wedge_diffraction_scene(), reference_frequency_hz=3.5e9);"
            "print('libwcmi.so' in open('/proc/self/maps').read(), 'libwcmi_host.so' in open('/proc/self/maps').read())")
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                         env={**os.environ, "PYTHONPATH": str(Path(compiler.__file__).resolve().parents[3])})
    assert run.stdout.split() == loaded, run.stdout + run.stderr


@pytest.mark.parametrize("call", ["call", "call_host"])
def test_native_entries_refuse_indices_outside_their_arrays(call):
    """The C entry points themselves, as a caller without the Python checks."""
    from witwin.channel import _native

    native = getattr(_native, call)
    welded, v = np.zeros((3, 3), np.int64), np.eye(3)
    zeros, base = np.zeros(1, np.int64), np.zeros(1, np.int64)
    ids = [np.zeros((3, k), np.int64) for k in (4, 6, 1)]
    count, offset, plane = np.zeros(1, np.int32), np.zeros(2, np.int32), np.array([[0.0, 0.0, 1.0, 0.0]])
    table, points = np.zeros(1, np.int32), np.zeros((6, 3))

    def edges(face):
        tri = np.array([face], np.int32)
        native("wc_edge_candidates", welded.ctypes.data, 3, tri.ctypes.data, 1, zeros.ctypes.data,
               base.ctypes.data, 1, table.ctypes.data, table.ctypes.data, *(a.ctypes.data for a in ids),
               count.ctypes.data)

    def hulls(face, first=(0, 1), listed=(0,)):
        tri, first, listed = (np.array(a, np.int32) for a in ([face], first, listed))
        native("wc_group_hulls", v.ctypes.data, 3, tri.ctypes.data, 1, first.ctypes.data, listed.ctypes.data,
               len(listed), plane.ctypes.data, 1, offset.ctypes.data, points.ctypes.data)

    edges([0, 1, 2])
    hulls([0, 1, 2])
    assert offset.tolist() == [0, 3]
    for face in ([0, 1, 3], [0, -4, 2]):
        with pytest.raises(RuntimeError, match="vertex"):
            edges(face)
        with pytest.raises(RuntimeError, match="vertex"):
            hulls(face)
    for first, listed in (((0, 2), (0,)), ((1, 0), (0,)), ((-1, 1), (0,))):
        with pytest.raises(RuntimeError, match="group"):
            hulls([0, 1, 2], first, listed)
    with pytest.raises(RuntimeError, match="face"):
        hulls([0, 1, 2], (0, 1), (1,))


def test_negative_face_and_vertex_ids_count_from_the_end():
    vertices, faces, _, _ = _random_mesh(2)
    n = len(faces)
    plane = np.tile([0.0, 0.6, 0.8, 0.3], (n, 1))
    a = compiler.group_hulls(vertices, faces, np.arange(n + 1), np.arange(n), plane)
    b = compiler.group_hulls(vertices, faces - len(vertices), np.arange(n + 1), np.arange(n) - n, plane)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_empty_mesh():
    none = np.zeros((0, 3), np.int32)
    edges, ev = compiler.build_edge_table(np.zeros((0, 3), np.float32), none, np.zeros(0, np.int32),
                                          np.zeros(0, np.int32))
    assert edges.shape == (0,) and ev.shape == (0, 4)
    offset, points = compiler.group_hulls(np.zeros((0, 3), np.float32), none, np.zeros(1, np.int32),
                                          np.zeros(0, np.int32), np.zeros((0, 4)))
    assert offset.tolist() == [0] and points.shape == (0, 3)


def test_group_hulls_keep_float64_vertices():
    """Corners are the vertices given: a few roundings of the in-plane basis on
    coordinates below 10 (1e-14), where single precision would move them 5e-7."""
    vertices = np.random.default_rng(3).uniform(-5.0, 5.0, (3, 3))
    n = np.cross(vertices[1] - vertices[0], vertices[2] - vertices[0])
    n /= np.linalg.norm(n)
    offset, points = compiler.group_hulls(vertices, np.array([[0, 1, 2]]), np.array([0, 1]), np.array([0]),
                                          np.append(n, n @ vertices[0])[None])
    assert offset.tolist() == [0, 3]
    assert np.abs(points[:, None] - vertices[None]).max(axis=2).min(axis=1).max() < 1e-14


def test_group_hulls_contain_their_faces():
    """Every hull runs counter-clockwise about its normal, holds its group's
    vertices (to 1e-9 of coordinates near 400 m) and has only them as corners."""
    c = compiler.compile(workloads.urban_canyon_scene(seed=2, shape=(2, 2)), reference_frequency_hz=3.5e9)
    offset, points = compiler.group_hulls(c.vertices, c.faces, c.group_face_offset, c.group_faces, c.group_plane)
    for g in range(c.group_count):
        hull = points[offset[g]:offset[g + 1]]
        members = c.group_faces[c.group_face_offset[g]:c.group_face_offset[g + 1]]
        pts = c.vertices[c.faces[members].reshape(-1)].astype(np.float64)
        n = c.group_plane[g, :3]
        assert 3 <= len(hull) <= len(np.unique(pts, axis=0))
        assert np.abs(hull[:, None] - pts[None]).max(axis=2).min(axis=1).max() < 1e-4  # off-plane part of a vertex
        for a, b in zip(hull, np.roll(hull, -1, axis=0)):
            assert (np.cross(b - a, pts - a) @ n >= -1e-9 * np.linalg.norm(b - a) * 400.0).all()


def test_scene_tables_count_their_own_changes():
    c = compiler.compile(workloads.urban_canyon_scene(seed=2, shape=(2, 2)), reference_frequency_hz=3.5e9)
    scene = compiler.DeviceScene(c, torch.device("cpu"))
    x = torch.ones(1, requires_grad=True)
    y = (x * scene.mat_eps).sum()
    scene.vertices.add_(1.0)
    y.backward()
    assert x.grad.item() == pytest.approx(float(scene.mat_eps.sum()))
    assert np.array_equal(scene.vertices.numpy(), c.vertices + np.float32(1.0))


def test_scene_hulls_are_those_of_the_uploaded_vertices():
    """Changing the compiled scene's arrays afterwards moves neither the device
    tables nor the hulls the chain culls bound their planes with."""
    c = compiler.compile(workloads.urban_canyon_scene(seed=2, shape=(2, 2)), reference_frequency_hz=3.5e9)
    want = compiler.DeviceScene(c, torch.device("cpu")).hulls()
    scene = compiler.DeviceScene(c, torch.device("cpu"))
    for table in (c.vertices, c.group_plane):
        table += 5.0
    for a, b in zip(scene.hulls(), want):
        assert torch.equal(a, b)
