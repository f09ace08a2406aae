"""GPU tests of the masked path export (wc_paths_count_masked /
wc_paths_emit_masked) against the per-cell export (wc_paths_count /
wc_paths_emit): the same kept rows in the same order, over every form of solve
the export takes (shared grids and per-transmitter sets, lane groups, either
visibility mode, each component alone, caps, single cells, no candidates)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from witwin.channel import workloads
from witwin.channel.components import component_bits
from witwin.channel.propagation import engine
from witwin.channel.scene.compiler import compile as compile_scene, device_scene
from witwin.core import Scene

pytestmark = pytest.mark.gpu

LRDT = ("los", "reflection", "diffraction", "transmission")
FORMS = [
    # tx, receivers per tx (None: one shared grid of 9 x 15), components, depth, cap, extra solve arguments
    pytest.param(1, None, LRDT, 3, None, {}, id="shared-grid"),
    pytest.param(3, None, LRDT, 2, 4, {}, id="shared-grid-3tx-cap"),
    pytest.param(3, (1, 64, 130), LRDT, 2, None, {}, id="uneven-sets"),
    pytest.param(3, (1, 64, 130), LRDT, 2, None, {"visibility_mode": 1}, id="uneven-sets-tile-loops"),
    pytest.param(2, (65, 7), LRDT, 2, None, {"lanes_per_cell": 4}, id="lane-groups"),
    pytest.param(1, (1,), LRDT, 1, None, {}, id="single-cell"),
    pytest.param(2, (33, 64), ("los",), 0, None, {}, id="los"),
    pytest.param(2, (33, 64), ("reflection",), 3, None, {}, id="reflection"),
    pytest.param(2, (33, 64), ("diffraction",), 1, 2, {}, id="diffraction-cap"),
    pytest.param(2, (33, 64), ("transmission",), 2, None, {"spatial_order": False}, id="transmission-plain-order"),
]


def _inputs(device, tx_count, rx_count, components, depth, extra, scene):
    rng = np.random.default_rng(17)
    compiled = compile_scene(scene, reference_frequency_hz=28.0e9)
    dscene = device_scene(compiled, device)
    up = lambda n: np.tile(np.array([[0.0, 0.0, 1.0]], np.float32), (n, 1))  # noqa: E731
    tx = workloads.street_points(rng, tx_count, z=(3.0, 30.0))
    if rx_count is None:
        gx, gy = np.meshgrid(np.linspace(1.3, 370.1, 9), np.linspace(2.9, 371.7, 15), indexing="ij")
        rx = np.stack([gx.ravel(), gy.ravel(), np.full(gx.size, 1.5)], axis=1).astype(np.float32)
        counts = None
    else:
        counts = np.asarray(rx_count)
        rx = workloads.street_points(rng, int(counts.sum()))
    inputs = engine.solve_inputs(compiled, dscene, components=component_bits(set(components)), max_depth=depth,
                                 coherent=True, frequency_hz=28.0e9, tx_pos=tx, tx_pol=up(tx_count),
                                 tx_power=np.linspace(0.5, 1.5, tx_count).astype(np.float32), rx_pos=rx,
                                 rx_pol=up(len(rx)), rx_count=counts, **extra)
    return dscene, inputs


def _both(monkeypatch, dscene, inputs, width, cap):
    masked = engine.export_rows(dscene, inputs, width=width, max_paths_per_pair=cap)
    assert engine.export_masks(dscene, inputs) is not None
    monkeypatch.setattr(engine, "EXPORT_MASK_LIMIT", 0)
    assert engine.export_masks(dscene, inputs) is None
    return masked, engine.export_rows(dscene, inputs, width=width, max_paths_per_pair=cap)


@pytest.mark.parametrize("tx_count,rx_count,components,depth,cap,extra", FORMS)
def test_masked_export_equals_per_cell_export(device, monkeypatch, tx_count, rx_count, components, depth, cap, extra):
    scene = workloads.batched_path_workload(tx_count=1).scene
    dscene, inputs = _inputs(device, tx_count, rx_count, components, depth, extra, scene)
    masked, plain = _both(monkeypatch, dscene, inputs, max(depth, 1), cap)
    assert set(masked) == set(plain)
    assert masked["dropped"] == plain["dropped"]
    for name, a in plain.items():
        if not isinstance(a, torch.Tensor):
            continue
        b = masked[name]
        assert a.shape == b.shape and a.dtype == b.dtype, name
        if a.is_floating_point() or a.is_complex():
            # the same device functions; one rounding apart where the compiler
            # contracts a multiply-add differently in the two kernels
            torch.testing.assert_close(b, a, rtol=2e-6, atol=1e-12, msg=lambda m: f"{name}: {m}")
        else:
            assert torch.equal(a, b), name


@pytest.mark.parametrize("rx_count,per_cell", [((1,), True), ((64,), True), ((65,), False)])
def test_both_exports_either_side_of_few_candidates(device, rx_count, per_cell):
    """Five chains over ten triangles: per cell up to 64 cells. The rows are the same either way."""
    from witwin.core import Mesh, PhysicalMaterial, Structure

    def wall(k):
        x, y = (80.0 * np.cos(k), 80.0 * np.sin(k))
        v = torch.tensor([[x, y, 0.0], [x - 30.0 * y / 80.0, y + 30.0 * x / 80.0, 0.0],
                          [x - 30.0 * y / 80.0, y + 30.0 * x / 80.0, 60.0], [x, y, 60.0]])
        return Structure(Mesh(v, torch.tensor([[0, 1, 2], [0, 2, 3]])), PhysicalMaterial(eps_r=4.0, sigma_e=0.01),
                         surface_id=k)

    scene = Scene(structures=[wall(k) for k in range(5)], endpoints=[])
    dscene, inputs = _inputs(device, 1, rx_count, ("los", "reflection", "transmission"), 1, {}, scene)
    assert inputs.view.max_tx_chains == 5 and dscene.view.face_count == 10
    assert engine._few_candidates(dscene, inputs) == per_cell
    masked = engine._export_rows(dscene, inputs, 1, None, [engine.export_masks(dscene, inputs)])
    plain = engine._export_rows(dscene, inputs, 1, None, [None])
    for name in ("tx_id", "rx_id", "component_id", "depth", "primitive_sequence"):
        assert torch.equal(masked[name], plain[name]), name
    torch.testing.assert_close(masked["path_field"], plain["path_field"], rtol=2e-6, atol=1e-12)


def test_masked_export_without_candidates(device, monkeypatch):
    dscene, inputs = _inputs(device, 2, (5, 70), ("los", "reflection"), 1, {}, Scene(structures=[], endpoints=[]))
    masked, plain = _both(monkeypatch, dscene, inputs, 1, None)
    assert masked["tx_id"].shape[0] == plain["tx_id"].shape[0] == 75
    assert torch.equal(masked["path_field"], plain["path_field"])
