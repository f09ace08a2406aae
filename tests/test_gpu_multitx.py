"""Several transmitters with their own scattered receiver sets in one launch
against one solve per transmitter: per-cell sums run in canonical order in
one lane, so every output of a cell is bit-identical whichever launch
evaluates it (the batched launch takes the per-transmitter-point-set paths of
the kernels, e.g. the queued edge visibility; the single solves the grid
paths)."""
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


def _say(msg: str) -> None:
    print(msg, flush=True)


def test_batched_transmitters_match_per_transmitter_solves(device):
    _say("case: 6 Tx with scattered street receivers (16..256 each), canyon, depth 2 + UTD + LoS, batched vs per Tx")
    compiled = compile_scene(workloads.urban_canyon_scene(seed=2, shape=(4, 4), spacing=2.0),
                             reference_frequency_hz=28e9)
    ds = device_scene(compiled, device)
    bits = component_bits({"los", "reflection", "diffraction"})
    tx_pos, sizes, rx_pos = workloads.batched_transmitters(seed=3, tx_count=6, max_rx=256)
    rx_pol = np.tile(np.array([[0, 0, 1]], np.float32), (rx_pos.shape[0], 1))
    tx_pol = np.tile(np.array([[0, 0, 1]], np.float32), (tx_pos.shape[0], 1))
    power = np.ones(tx_pos.shape[0], np.float32)
    batched = engine.solve_inputs(compiled, ds, components=bits, max_depth=2, coherent=True, frequency_hz=28e9,
                                  tx_pos=tx_pos, tx_pol=tx_pol, tx_power=power, rx_pos=rx_pos, rx_pol=rx_pol,
                                  rx_count=sizes)
    assert int(batched.view.rx_shared) == 0
    out = engine.radiomap_forward(ds, batched)
    torch.cuda.synchronize()
    names = ("power_total", "field_total", "component_power", "component_field", "diffraction_vector", "path_count")
    got = {k: getattr(out, k).cpu().numpy() for k in names}
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    total_paths = 0
    for t in range(tx_pos.shape[0]):
        sl = slice(int(offsets[t]), int(offsets[t + 1]))
        single = engine.solve_inputs(compiled, ds, components=bits, max_depth=2, coherent=True, frequency_hz=28e9,
                                     tx_pos=tx_pos[t:t + 1], tx_pol=tx_pol[t:t + 1], tx_power=power[t:t + 1],
                                     rx_pos=rx_pos[sl], rx_pol=rx_pol[sl])
        ref = engine.radiomap_forward(ds, single)
        torch.cuda.synchronize()
        for k in names:
            want = getattr(ref, k).cpu().numpy()
            have = got[k][..., sl] if k.startswith("component") else got[k][sl]
            np.testing.assert_array_equal(have, want, err_msg=f"tx {t} {k}")
        total_paths += int(ref.path_count.sum().item())
    _say(f"cells {int(sizes.sum())}, paths {total_paths}")
    assert total_paths > 0


@pytest.mark.parametrize("tx_count,receivers", [(8, 5), (64, 3), (64, 512)],
                         ids=["tree-walk", "no-table", "tree-walk-many-receivers"])
def test_edge_shadows_do_not_change_the_map(device, tx_count, receivers):
    """Terrain of 8,058 triangles with every edge diffracting (12,149): one
    transmitter's shadow table comes from all triangles, eight transmitters' from
    the tree, 64 transmitters' only where each has many receivers. The cells of
    one transmitter are the same bits in all of them."""
    terrain = workloads.heightfield_scene(seed=4, size=64, boxes=10, shape=(2, 2))
    scene = Scene(structures=list(terrain.structures), endpoints=list(terrain.endpoints))
    compiled = compile_scene(scene, reference_frequency_hz=3.5e9)
    ds = device_scene(compiled, device)
    assert compiled.face_count == 8058 and compiled.edge_count == 12149
    rng = np.random.default_rng(8)
    top = float(compiled.vertices[:, 2].max())
    tx = np.concatenate([rng.uniform(20.0, 106.0, (tx_count, 2)), rng.uniform(top - 8.0, top + 6.0, (tx_count, 1))], 1)
    n = tx_count * receivers
    rx = np.concatenate([rng.uniform(2.0, 124.0, (n, 2)), rng.uniform(top - 10.0, top + 2.0, (n, 1))], 1)
    tx, rx = tx.astype(np.float32), rx.astype(np.float32)
    up = lambda k: np.tile(np.array([[0, 0, 1]], np.float32), (k, 1))  # noqa: E731

    def solve(t, r, counts):
        inputs = engine.solve_inputs(compiled, ds, components=component_bits({"los", "diffraction"}), max_depth=1,
                                     coherent=True, frequency_hz=3.5e9, tx_pos=t, tx_pol=up(len(t)),
                                     tx_power=np.ones(len(t), np.float32), rx_pos=r, rx_pol=up(len(r)),
                                     rx_count=counts)
        out = engine.radiomap_forward(ds, inputs)
        torch.cuda.synchronize()
        return {k: getattr(out, k).cpu().numpy() for k in ("power_total", "field_total", "path_count")}

    _say(f"case: {tx_count} transmitters x {receivers} receivers, 12,149 edges")
    got = solve(tx, rx, np.full(tx_count, receivers))
    for t in (0, tx_count - 1):
        sl = slice(t * receivers, (t + 1) * receivers)
        want = solve(tx[t:t + 1], rx[sl], np.array([receivers]))
        assert want["path_count"].max() > 100
        for k in want:
            np.testing.assert_array_equal(got[k][sl], want[k], err_msg=f"tx {t} {k}")
