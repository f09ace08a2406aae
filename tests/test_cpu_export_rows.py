"""The masked path export's row kernels checked on the CPU (device sources
compiled as host C++ through a shim): a row whose dealt candidate the evaluating
kernel does not find again, which two differently compiled kernels may disagree
on at a wall or a face border within rounding. Its interactions come from the
kernel that evaluates it, and where there are none the row is absent under an
identity no real row has."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_cpu_culls import _build, _run
from test_cpu_oracle_and_host import _sah_tables
from witwin.channel import workloads
from witwin.channel.scene.compiler import compile as compile_scene
from witwin.core import Mesh, PhysicalMaterial, Scene, Structure


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    def wall(k, x):
        v = torch.tensor([[x, -40.0, -40.0], [x, 40.0, -40.0], [x, 40.0, 40.0], [x, -40.0, 40.0]])
        return Structure(Mesh(v, torch.tensor([[0, 1, 2], [0, 2, 3]])), PhysicalMaterial(eps_r=4.0, sigma_e=0.01),
                         surface_id=k)

    scene = Scene(structures=[wall(k, 10.0 * (k + 1)) for k in range(3)],
                  endpoints=[workloads.transmitter((0.0, 0.0, 1.0)), workloads.receiver((0.0, 1.0, 1.0))])
    compiled = compile_scene(scene, reference_frequency_hz=3.5e9)
    assert compiled.group_count == 3
    nodes, sorted_tris, face_tris = _sah_tables(compiled)
    out = tmp_path_factory.mktemp("export")
    nodes.tofile(out / "nodes.bin")
    sorted_tris.astype(np.float32).tofile(out / "tris.bin")
    face_tris.astype(np.float32).tofile(out / "ftris.bin")
    compiled.group_plane.astype(np.float64).tofile(out / "plane.bin")
    compiled.group_face_offset.astype(np.int32).tofile(out / "goff.bin")
    compiled.group_faces.astype(np.int32).tofile(out / "gfaces.bin")
    return _run(_build(tmp_path_factory, "export_rows_check"), out)


def test_straight_row_follows_the_walls_its_kernel_finds(report):
    assert report["straight"] == 120 and report["gone"] > 0
    assert report["straight_wrong"] == 0


def test_chain_without_hits_leaves_an_absent_row(report):
    assert report["chains"] == report["chains_right"] == 10
