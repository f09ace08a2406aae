"""Timed cases of the propagation framework: what a user's program calls, over
the range of sizes it is called with.

Each case is a plain dict with a ``kind`` and its sizes. ``prepare`` builds what
a program holds before the call (scenes, compiled scenes, plans, endpoint
tensors) from a seed, ``run`` makes one call through the public entry points,
``exact`` restates the result in 64 bits with plain torch where it has a closed
form. Geometry comes from the seeded workloads of ``witwin.channel.workloads``;
the seed of a preparation moves the transmitters and receivers (and the row
tables), as a program that sweeps positions through one environment does.
"""

from __future__ import annotations

import functools
import math
import sys
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch
from torch.autograd import forward_ad

_PACKAGE = str(Path(__file__).resolve().parent.parent / "witwin-channel_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from witwin.channel import deterministic, path, workloads  # noqa: E402
from witwin.channel.components import component_bits  # noqa: E402
from witwin.channel.kernels.deterministic import MeanDbStep  # noqa: E402
from witwin.channel.kernels.fields import field_reflection_sequence_ad  # noqa: E402
from witwin.channel.propagation import batching, consumer, engine  # noqa: E402
from witwin.channel.scene.compiler import compile as compile_scene, device_scene  # noqa: E402
from witwin.core import AntennaState, PhysicalMaterial, Scene  # noqa: E402

C0 = 299792458.0
EPS0 = 8.8541878128e-12
LRD = "los,reflection,diffraction"
LRDT = "los,reflection,diffraction,transmission"


# ---------------------------------------------------------------- cases

def listed():
    return [
        # a link check: transmitter over a ground plane, a small receiver grid, 3.5 GHz. The whole call is
        # latency: scene compile, planning, launches, result assembly
        dict(name="two_ray_map", kind="two_ray", rows=16, cols=16, frequency=3.5e9),
        # one coverage map of a city block through the public solver: 256 x 256 cells, three bounces and edge
        # diffraction at 28 GHz, from a Scene to the result tensors
        dict(name="canyon_map", kind="map", rows=256, cols=256, depth=3, components=LRD, ad="none",
             frequency=28.0e9),
        # the same map differentiated: solve(ad_mode="vjp"), a mean-dB loss, backward to the transmitter position
        dict(name="canyon_map_vjp", kind="map", rows=256, cols=256, depth=3, components=LRD, ad="vjp",
             frequency=28.0e9),
        # a calibration loop's step on a held plan: forward and adjoint of the mean-dB loss, captured and replayed
        dict(name="canyon_step", kind="step", rows=256, cols=256, depth=3, components=LRD, frequency=28.0e9),
        # the same step for many transmitters with uneven sets of street receivers (16 to 4,096 each)
        dict(name="street_points_step", kind="points", tx=64, rx_min=16, rx_max=4096, depth=3, components=LRD,
             frequency=28.0e9),
        # terrain calibration: 32,738 triangles, depth-2 reflection, gradient with respect to every vertex too
        dict(name="terrain_vertex_step", kind="terrain", rows=256, cols=256, depth=2, frequency=3.5e9),
        # the large batched step: 134,850 triangles, 8 materials, five bounces, diffraction and transmission at two
        # carriers, transmitters with receiver grids from 64^2 to 512^2
        dict(name="city_batch_step", kind="city", tx=8, side_min=64, side_max=512, depth=5, components=LRDT),
        # explicit path rows of many transmitters with their own receiver sets (layered walls on the streets)
        dict(name="street_paths", kind="paths", tx=64, rx_min=16, rx_max=4096, depth=3, components=LRDT,
             frequency=28.0e9),
        # channel frequency responses of padded path sets on an OFDM grid
        dict(name="subcarrier_response", kind="cfr", pairs=45221, paths=199, mean_paths=18.0, subcarriers=1024,
             bandwidth=100.0e6, frequency=28.0e9, normalize=False),
        # the consumer interface discovering 32 sources x 32 sinks, line of sight and single reflections
        dict(name="consumer_discovery", kind="discover", sources=32, sinks=32, depth=1, components="los,reflection",
             frequency=28.0e9),
        # time-varying replay: the rows of a frozen discovery re-evaluated at 64 time slots' moved endpoints
        dict(name="consumer_replay", kind="replay", sources=16, sinks=16, slots=64, depth=2,
             components="los,reflection", frequency=28.0e9),
        # the row operators of a training program: three-bounce Jones transport of explicit rows, forward and backward
        dict(name="reflection_rows", kind="rows", count=262144, depth=3, frequency=28.0e9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["two_ray", "map", "map", "step", "points", "terrain", "city", "paths", "cfr", "discover",
                       "replay", "rows"])
    carrier = rng.choice([2.4e9, 3.5e9, 28.0e9])
    if kind == "two_ray":
        return dict(kind=kind, rows=_log(rng, 1, 64), cols=_log(rng, 1, 64), frequency=carrier)
    if kind == "map":
        return dict(kind=kind, rows=_log(rng, 9, 256), cols=_log(rng, 9, 256), depth=rng.randint(1, 3),
                    components=rng.choice([LRD, "los,diffraction", "los,reflection"]), ad=rng.choice(["none", "vjp", "jvp"]),
                    frequency=carrier)
    if kind == "step":
        return dict(kind=kind, rows=_log(rng, 9, 256), cols=_log(rng, 9, 256), depth=rng.randint(1, 3),
                    components=rng.choice([LRD, "los,diffraction", "los,reflection"]), frequency=carrier)
    if kind in ("points", "paths"):
        lo = _log(rng, 1, 64)
        return dict(kind=kind, tx=_log(rng, 1, 64), rx_min=lo, rx_max=max(lo, _log(rng, 64, 4096)),
                    depth=rng.randint(1, 3), components=rng.choice([LRD, LRDT]), frequency=carrier)
    if kind == "terrain":
        return dict(kind=kind, rows=_log(rng, 17, 256), cols=_log(rng, 17, 256), depth=rng.randint(1, 2),
                    frequency=rng.choice([2.4e9, 3.5e9]))
    if kind == "city":
        return dict(kind=kind, tx=rng.randint(1, 6), side_min=rng.randint(33, 64), side_max=rng.randint(65, 512),
                    depth=rng.randint(2, 5), components=rng.choice([LRDT, LRD]))
    if kind == "cfr":
        mean = rng.uniform(2.0, 18.0)
        return dict(kind=kind, pairs=_log(rng, 64, 45221), paths=_log(rng, 20, 199), mean_paths=round(mean, 2),
                    subcarriers=_log(rng, 48, 1024), bandwidth=rng.choice([20.0e6, 100.0e6]), frequency=carrier,
                    normalize=rng.random() < 0.5)
    if kind == "discover":
        return dict(kind=kind, sources=_log(rng, 1, 32), sinks=_log(rng, 1, 256), depth=rng.randint(1, 3),
                    components=rng.choice(["los,reflection", LRD]), frequency=carrier)
    if kind == "replay":
        return dict(kind=kind, sources=_log(rng, 1, 16), sinks=_log(rng, 4, 64), slots=_log(rng, 1, 64),
                    depth=rng.randint(1, 3), components="los,reflection", frequency=carrier)
    return dict(kind=kind, count=_log(rng, 1000, 262144), depth=rng.randint(1, 5), frequency=carrier)


# ---------------------------------------------------------------- environments a program holds

def _device():
    return torch.device("cuda", torch.cuda.current_device())


@functools.lru_cache(maxsize=None)
def _canyon_structures():
    """Structures of the urban canyon (seed 2: 64 boxes and the ground)."""
    return tuple(workloads.urban_canyon_scene(seed=2, shape=(2, 2)).structures)


@functools.lru_cache(maxsize=None)
def _canyon(frequency):
    scene = workloads.urban_canyon_scene(seed=2, shape=(2, 2))
    return compile_scene(scene, reference_frequency_hz=frequency)


@functools.lru_cache(maxsize=None)
def _walled_canyon(frequency):
    """The canyon with the three layered street walls."""
    scene = workloads.urban_canyon_scene(seed=2, shape=(2, 2))
    walls = [workloads.street_wall(*seg, h, layers, 900 + k)
             for k, (seg, h, layers) in enumerate(workloads.STREET_WALLS)]
    scene = Scene(structures=list(scene.structures) + walls, endpoints=list(scene.endpoints))
    return compile_scene(scene, reference_frequency_hz=frequency)


@functools.lru_cache(maxsize=None)
def _terrain(frequency):
    scene = workloads.heightfield_scene(seed=4, shape=(2, 2))
    top = max(float(s.geometry.vertices[:, 2].max()) for s in scene.structures[:1])
    return compile_scene(scene, reference_frequency_hz=frequency), top


@functools.lru_cache(maxsize=None)
def _city():
    """The 400-box city on a 256 x 256 heightfield and 256 transmitter sites."""
    w = workloads.scaled_city(seed=5, tx_count=256, side_range=(2, 2))
    return w, compile_scene(w.scene, reference_frequency_hz=w.frequencies[0])


CANYON_EXTENT = 15.0 + 8 * 45.0


def _canyon_grid(rows, cols):
    """Receiver grid 1.5 m high over the canyon; (origin, spacing) as the canyon workload places its 256 x 256."""
    spacing = 510.0 / max(rows - 1, cols - 1, 1)
    origin = ((CANYON_EXTENT - (rows - 1) * spacing) / 2.0 + 0.173,
              (CANYON_EXTENT - (cols - 1) * spacing) / 2.0 + 0.291, 1.5)
    return origin, spacing


def _grid_points(origin, rows, cols, spacing):
    gx, gy = np.meshgrid(np.arange(rows, dtype=np.float32), np.arange(cols, dtype=np.float32), indexing="ij")
    pts = np.stack([origin[0] + spacing * gx.reshape(-1), origin[1] + spacing * gy.reshape(-1),
                    np.full(rows * cols, origin[2])], axis=1)
    return pts.astype(np.float32)


def _up(n):
    return np.tile(np.array([[0.0, 0.0, 1.0]], np.float32), (n, 1))


def _tilted(rng, n):
    """Antenna axes up to a few degrees off vertical."""
    v = rng.normal(0.0, 0.05, (n, 3)) + np.array([0.0, 0.0, 1.0])
    return (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)


def _upright(rng, n):
    """Vertical antenna axes, mounted either way up."""
    return ((rng.integers(0, 2, (n, 1)) * 2 - 1) * _up(n)).astype(np.float32)


def _sites(case):
    """Generator of the positions a case's sizes fix."""
    return np.random.default_rng([int(v) for v in case.values() if isinstance(v, (int, float))])


def _set_sizes(case):
    """Uneven receiver-set sizes, evenly spread over the logarithm of [rx_min, rx_max]."""
    t = case["tx"]
    u = (np.arange(t) + 0.5) / t
    sizes = np.exp(np.log(case["rx_min"]) + u * (np.log(case["rx_max"]) - np.log(case["rx_min"])))
    return np.maximum(np.floor(sizes).astype(np.int64), 1)


def _components(case):
    return set(case["components"].split(","))


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_two_ray(case, seed):
    rng = np.random.default_rng(seed)
    rows, cols = case["rows"], case["cols"]
    ground = PhysicalMaterial(eps_r=5.31, sigma_e=0.0326, thickness_m=5.0, name="ground")
    tx = (float(rng.uniform(-5.0, 5.0)), float(rng.uniform(-5.0, 5.0)), float(rng.uniform(6.0, 14.0)))
    origin = (-(rows - 1) / 2.0 + 0.25, -(cols - 1) / 2.0 + 0.25, 1.5)
    scene = Scene(structures=[workloads.ground_structure(-1.0e4, -1.0e4, 1.0e4, 1.0e4, ground)],
                  endpoints=[workloads.transmitter(tx), workloads.grid(origin, (rows, cols), 1.0)])
    config = deterministic.Config(components={"los", "reflection"}, max_depth=1)
    return SimpleNamespace(kind="two_ray", scene=scene, config=config, frequency=case["frequency"], tx=tx,
                           origin=origin)


def _prepare_map(case, seed):
    rng = np.random.default_rng(seed)
    tx = workloads.street_points(rng, 1, z=(3.0, 30.0))[0]
    origin, spacing = _canyon_grid(case["rows"], case["cols"])
    scene = Scene(structures=list(_canyon_structures()),
                  endpoints=[workloads.transmitter(tuple(map(float, tx))),
                             workloads.grid(origin, (case["rows"], case["cols"]), spacing)])
    config = deterministic.Config(components=_components(case), max_depth=case["depth"], ad_mode=case["ad"])
    if case["ad"] == "vjp":
        scene.endpoints[0].position.requires_grad_(True)
    return SimpleNamespace(kind="map", scene=scene, config=config, frequency=case["frequency"], ad=case["ad"],
                           direction=torch.tensor([0.6, -0.64, 0.48]))


def _prepare_step(case, seed):
    rng = np.random.default_rng(seed)
    compiled = _canyon(case["frequency"])
    dscene = device_scene(compiled, _device())
    tx = workloads.street_points(rng, 1, z=(3.0, 30.0))
    origin, spacing = _canyon_grid(case["rows"], case["cols"])
    rx = _grid_points(origin, case["rows"], case["cols"], spacing)
    inputs = engine.solve_inputs(compiled, dscene, components=component_bits(_components(case)),
                                 max_depth=case["depth"], coherent=True, frequency_hz=case["frequency"], tx_pos=tx,
                                 tx_pol=_up(1), tx_power=np.ones(1, np.float32), rx_pos=rx, rx_pol=_up(len(rx)))
    step = MeanDbStep(dscene, inputs, compiled.materials.count)
    step.capture()
    return SimpleNamespace(kind="step", step=step)


def _prepare_points(case, seed):
    rng = np.random.default_rng(seed)
    compiled = _canyon(case["frequency"])
    dscene = device_scene(compiled, _device())
    t = case["tx"]
    tx = workloads.street_points(rng, t, z=(3.0, 30.0))
    count = rng.permutation(_set_sizes(case))
    rx = workloads.street_points(rng, int(count.sum()))
    inputs = engine.solve_inputs(compiled, dscene, components=component_bits(_components(case)),
                                 max_depth=case["depth"], coherent=True, frequency_hz=case["frequency"], tx_pos=tx,
                                 tx_pol=_up(t), tx_power=np.ones(t, np.float32), rx_pos=rx, rx_pol=_up(len(rx)),
                                 rx_count=count)
    step = MeanDbStep(dscene, inputs, compiled.materials.count)
    step.capture()
    return SimpleNamespace(kind="step", step=step)


def _prepare_terrain(case, seed):
    rng = np.random.default_rng(seed)
    compiled, top = _terrain(case["frequency"])
    dscene = device_scene(compiled, _device())
    extent = 127 * 2.0
    tx = np.array([[rng.uniform(60.0, extent - 60.0), rng.uniform(60.0, extent - 60.0),
                    top + rng.uniform(20.0, 30.0)]], np.float32)
    spacing = extent / max(case["rows"], case["cols"])
    origin = ((extent - (case["rows"] - 1) * spacing) / 2.0 + 0.137,
              (extent - (case["cols"] - 1) * spacing) / 2.0 + 0.219, top + 1.5)
    rx = _grid_points(origin, case["rows"], case["cols"], spacing)
    inputs = engine.solve_inputs(compiled, dscene, components=component_bits({"los", "reflection"}),
                                 max_depth=case["depth"], coherent=True, frequency_hz=case["frequency"], tx_pos=tx,
                                 tx_pol=_up(1), tx_power=np.ones(1, np.float32), rx_pos=rx, rx_pol=_up(len(rx)))
    step = MeanDbStep(dscene, inputs, compiled.materials.count, vertices=True)
    step.capture()
    return SimpleNamespace(kind="step", step=step)


def _prepare_city(case, seed):
    rng = np.random.default_rng(seed)
    w, compiled = _city()
    dscene = device_scene(compiled, _device())
    t = case["tx"]
    sites = w.tx[rng.choice(w.tx.shape[0], t, replace=False)]
    sides = np.exp(np.linspace(math.log(case["side_min"]), math.log(case["side_max"]), t))
    sides = rng.permutation(np.round(sides).astype(np.int64)) if t > 1 else np.array([case["side_max"]], np.int64)
    rx = []
    for s in sides:
        spacing = w.extent / float(s)
        rx.append(_grid_points((0.5 * spacing, 0.5 * spacing, w.receiver_z), int(s), int(s), spacing))
    run = batching.BatchedMeanDb(compiled, dscene, sites, np.concatenate(rx), sides * sides,
                                 components=component_bits(_components(case)), max_depth=case["depth"],
                                 frequencies=w.frequencies, shape=batching.LaunchShape(1, 16))
    run.capture()
    return SimpleNamespace(kind="city", run=run)


def _prepare_paths(case, seed):
    """Sites fixed by the case's sizes (so that the number of rows is), their order and antennas by the seed."""
    rng, sites = np.random.default_rng(seed), _sites(case)
    compiled = _walled_canyon(case["frequency"])
    dscene = device_scene(compiled, _device())
    t = case["tx"]
    tx = workloads.street_points(sites, t, z=(3.0, 30.0))
    count = sites.permutation(_set_sizes(case))
    rx = np.split(workloads.street_points(sites, int(count.sum())), np.cumsum(count)[:-1])
    order = rng.permutation(t)
    tx, count, rx = tx[order], count[order], np.concatenate([rng.permutation(rx[i]) for i in order])
    comps = _components(case)
    inputs = engine.solve_inputs(compiled, dscene, components=component_bits(comps), max_depth=case["depth"],
                                 coherent=True, frequency_hz=case["frequency"], tx_pos=tx, tx_pol=_upright(rng, t),
                                 tx_power=np.ones(t, np.float32), rx_pos=rx, rx_pol=_upright(rng, len(rx)),
                                 rx_count=count)
    return SimpleNamespace(kind="paths", compiled=compiled, dscene=dscene, inputs=inputs, tx=tx, rx=rx, count=count,
                           config=path.Config(components=comps, max_depth=case["depth"]))


def _prepare_cfr(case, seed):
    """Padded path sets: a strong first path, later ones weaker; sizes geometric about ``mean_paths``, the largest
    filling the padding, as in the batched street solve."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    b, p = case["pairs"], case["paths"]
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    count = torch.clamp((-case["mean_paths"] * torch.log(1.0 - 0.999 * rand(b))).to(torch.int64), 1, p)
    count[0] = p
    valid = torch.arange(p, device="cuda").view(1, -1) < count.view(-1, 1)
    first = (5.0 + 295.0 * rand(b, 1)) / C0
    tau = first + torch.cumsum(rand(b, p) * (20.0 / C0), dim=1)
    tau = torch.where(valid, tau, torch.zeros_like(tau)).to(torch.float32)
    mag = 1.0e-5 * torch.exp(-3.0 * rand(b, p)) / (1.0 + torch.arange(p, device="cuda"))
    a = torch.polar(mag, 2.0 * math.pi * rand(b, p))
    a = torch.where(valid, a, torch.zeros_like(a)).to(torch.complex64).unsqueeze(-1).contiguous()
    k = torch.arange(case["subcarriers"], dtype=torch.float64)
    spacing = case["bandwidth"] / case["subcarriers"]
    freqs = case["frequency"] + (k - case["subcarriers"] // 2) * spacing
    return SimpleNamespace(kind="cfr", a=a, tau=tau, valid=valid, freqs=freqs, normalize=case["normalize"])


def _batch(points, polarizations, device, powers=None):
    n = len(points)
    return consumer.EndpointBatch(
        stable_ids=torch.arange(1, n + 1, dtype=torch.int64, device=device),
        positions_m=torch.as_tensor(points, dtype=torch.float32, device=device).contiguous(),
        polarizations=torch.as_tensor(polarizations, device=device),
        powers_w=None if powers is None else torch.as_tensor(powers.astype(np.float32), device=device))


def _discovery(case):
    """Sources and sinks fixed by the case's sizes (so that the number of rows is)."""
    sites = _sites(case)
    sources = workloads.street_points(sites, case["sources"], z=(3.0, 30.0))
    sinks = workloads.street_points(sites, case["sinks"])
    return _canyon(case["frequency"]), sources, sinks


def _request(case, sources, sinks):
    return consumer.PropagationRequest(
        sources=sources, sinks=sinks, reference_frequency_hz=case["frequency"],
        components=frozenset(_components(case)), max_depth=case["depth"], response="scalar_transport",
        topology_mode="discover", ad_mode="none")


def _prepare_discover(case, seed):
    rng = np.random.default_rng(seed)
    compiled, sources, sinks = _discovery(case)
    device = _device()
    device_scene(compiled, device)
    sources, sinks = rng.permutation(sources), rng.permutation(sinks)
    request = _request(case, _batch(sources, _upright(rng, len(sources)), device, np.ones(len(sources))),
                       _batch(sinks, _upright(rng, len(sinks)), device))
    return SimpleNamespace(kind="discover", compiled=compiled, request=request)


def _prepare_replay(case, seed):
    rng = np.random.default_rng(seed)
    compiled, sources, sinks = _discovery(case)
    device = _device()
    found = consumer.evaluate(compiled, _request(case, _batch(sources, _up(len(sources)), device, np.ones(len(sources))),
                                                 _batch(sinks, _up(len(sinks)), device)))
    prepared = consumer.prepare_fixed_topology(found.paths.topology)
    slots = case["slots"]
    tiled = consumer.replicate_over_slots(prepared, slots, source_count=case["sources"], sink_count=case["sinks"])
    # sinks drift up to 0.3 m per axis over the slots
    drift = np.linspace(0.0, 1.0, slots)[:, None, None] * rng.uniform(-0.3, 0.3, (1, case["sinks"], 3))
    moved = (sinks[None] + drift).reshape(-1, 3).astype(np.float32)
    request = consumer.FixedTopologyRequest(
        sources=_batch(np.tile(sources, (slots, 1)), _tilted(rng, slots * len(sources)), device,
                       rng.uniform(0.1, 2.0, slots * len(sources))),
        sinks=_batch(moved, _tilted(rng, len(moved)), device),
        reference_frequency_hz=case["frequency"], topology=tiled, response="scalar_transport", ad_mode="none",
        slot_count=slots)
    return SimpleNamespace(kind="replay", compiled=compiled, request=request)


_ROW_NAMES = ("source", "target", "positions", "normals", "power", "tx_pol", "rx_pol", "eps", "sigma", "mu", "gain",
              "thickness")
_ROW_GRADS = ("source", "target", "positions", "normals", "eps", "sigma")


def _prepare_rows(case, seed):
    """Rows of a training program: interaction points spread over a street canyon, wall materials of the canyon and
    the city, gradients to endpoints, points, normals and materials."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, d = case["count"], case["depth"]
    uni = lambda lo, hi, *s: lo + (hi - lo) * torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    source = torch.stack([uni(0.0, 360.0, n), uni(0.0, 360.0, n), uni(3.0, 30.0, n)], dim=1)
    target = torch.stack([uni(0.0, 360.0, n), uni(0.0, 360.0, n), torch.full((n,), 1.5, device="cuda")], dim=1)
    positions = torch.stack([uni(0.0, 360.0, n, d), uni(0.0, 360.0, n, d), uni(0.0, 30.0, n, d)], dim=2)
    normals = torch.nn.functional.normalize(uni(-1.0, 1.0, n, d, 3), dim=-1)
    table = torch.tensor([[5.31, 0.0326, 0.2], [6.27, 0.0043, 0.02], [3.75, 0.038, 0.25], [1.99, 0.0047, 0.05]],
                         device="cuda")
    mats = table[torch.randint(0, 4, (n, d), generator=g, device="cuda")]
    pol = torch.tensor([0.0, 0.0, 1.0], device="cuda").expand(n, 3).contiguous()
    t = dict(source=source, target=target, positions=positions, normals=normals, power=uni(0.1, 2.0, n), tx_pol=pol,
             rx_pol=pol.clone(), eps=mats[..., 0].contiguous(), sigma=mats[..., 1].contiguous(),
             mu=torch.ones(n, d, device="cuda"), gain=torch.ones(n, d, device="cuda"),
             thickness=mats[..., 2].contiguous())
    t = {k: v.to(torch.float32).contiguous() for k, v in t.items()}
    for k in _ROW_GRADS:
        t[k].requires_grad_(True)
    weight = torch.complex(uni(-1.0, 1.0, n), uni(-1.0, 1.0, n)).to(torch.complex64)
    return SimpleNamespace(kind="rows", t=t, weight=weight, frequency=case["frequency"])


_PREPARE = {"two_ray": _prepare_two_ray, "map": _prepare_map, "step": _prepare_step, "points": _prepare_points,
            "terrain": _prepare_terrain, "city": _prepare_city, "paths": _prepare_paths, "cfr": _prepare_cfr,
            "discover": _prepare_discover, "replay": _prepare_replay, "rows": _prepare_rows}


# ---------------------------------------------------------------- run

def run(state):
    return _RUN[state.kind](state)


def _run_two_ray(s):
    r = deterministic.solve(s.scene, s.config, reference_frequency_hz=s.frequency)
    return {"path_gain": r.path_gain, "field": r.field, "los": r.component_power["los"],
            "reflection": r.component_power["reflection"], "los_field": r.component_fields["los"],
            "reflection_field": r.component_fields["reflection"]}


def _map_outputs(r):
    out = {"path_gain": r.path_gain, "field": r.field}
    out.update({f"power_{k}": v for k, v in r.component_power.items()})
    out.update({f"field_{k}": v for k, v in r.component_fields.items()})
    return out


def _mean_db(power):
    lit = power > 0
    db = 10.0 * torch.log10(torch.where(lit, power, torch.ones_like(power)))
    return db.sum() / lit.sum().clamp_min(1)


def _run_map(s):
    tx = s.scene.endpoints[0]
    if s.ad == "vjp":
        tx.position.grad = None
        r = deterministic.solve(s.scene, s.config, reference_frequency_hz=s.frequency)
        _mean_db(r.path_gain).backward()
        return {**{k: v.detach() for k, v in _map_outputs(r).items()}, "grad_tx": tx.position.grad}
    if s.ad == "jvp":
        with forward_ad.dual_level():
            moving = AntennaState(tx.antenna_id, "tx", forward_ad.make_dual(tx.position, s.direction))
            scene = Scene(structures=s.scene.structures, endpoints=[moving, s.scene.endpoints[1]])
            r = deterministic.solve(scene, s.config, reference_frequency_hz=s.frequency)
            value, tangent = forward_ad.unpack_dual(r.path_gain)
        return {"path_gain": value, "path_gain_tangent": tangent}
    return _map_outputs(deterministic.solve(s.scene, s.config, reference_frequency_hz=s.frequency))


def _step_outputs(step):
    o = step.out
    out = {"power": o.power_total, "field": o.field_total, "component_power": o.component_power,
           "component_field": o.component_field, "paths": o.path_count, "grad_params": step.grad_params,
           "grad_tx": step.grad_tx}
    if step.vertices:
        out["grad_vertices"] = step.grad_vertices
    return out


def _run_step(s):
    s.step.step()
    return _step_outputs(s.step)


def _run_city(s):
    s.run.step()
    out = {"grad_params": s.run.grad_params, "grad_frequency": s.run.grad_frequency, "grad_tx": s.run.grad_tx}
    for k, (fi, _, step) in enumerate(s.run.units):
        out[f"power_{k}"] = step.out.power_total
        out[f"field_{k}"] = step.out.field_total
        out[f"paths_{k}"] = step.out.path_count
    return out


def _run_paths(s):
    p = path.solve_batched(s.compiled, s.config, s.tx, s.rx, s.count, dscene=s.dscene, inputs=s.inputs)
    out = {f"row_{k}": v for k, v in p.rows.items() if isinstance(v, torch.Tensor)}
    out.update(pair_offset=p.pair_offset, pair_tx=p.pair_tx, pair_rx=p.pair_rx, theta_t=p.theta_t, phi_t=p.phi_t,
               theta_r=p.theta_r, phi_r=p.phi_r)
    return out


def _run_cfr(s):
    return path.paths_cfr(s.a, s.tau, s.valid, s.freqs, normalize_delays=s.normalize)


def _batch_outputs(paths):
    t, g = paths.topology, paths.geometry
    return {"pair_index": paths.pair_index, "pair_offsets": paths.pair_offsets, "depth": t.depth,
            "component": t.component_id, "primitives": t.primitive_sequence, "materials": t.material_sequence,
            "edge": t.edge_id, "interaction": t.interaction_type, "length": g.path_length_m, "delay": g.delay_s,
            "direction": g.field_direction, "positions": g.interaction_positions_m,
            "normals": g.interaction_normals, "coefficient": paths.transport.coefficient}


def _run_discover(s):
    return _batch_outputs(consumer.evaluate(s.compiled, s.request).paths)


def _run_replay(s):
    r = consumer.reevaluate(s.compiled, s.request)
    return {**_batch_outputs(r.paths), "row_valid": r.row_valid}


def _run_rows(s):
    t = s.t
    out = field_reflection_sequence_ad(*(t[k] for k in _ROW_NAMES), frequency=s.frequency)
    inputs = [t[k] for k in _ROW_GRADS]
    grads = torch.autograd.grad(out["path_field"], inputs, grad_outputs=s.weight)
    res = {k: out[k].detach() for k in ("field_vector", "coefficient", "path_field", "path_gain", "path_length_m",
                                        "delay_s", "direction")}
    res.update({f"grad_{k}": g for k, g in zip(_ROW_GRADS, grads)})
    return res


_RUN = {"two_ray": _run_two_ray, "map": _run_map, "step": _run_step, "city": _run_city, "paths": _run_paths,
        "cfr": _run_cfr, "discover": _run_discover, "replay": _run_replay, "rows": _run_rows}


# ---------------------------------------------------------------- work

# arithmetic a path cannot do without, from counting the formulas: slab coefficients and Jones step of one
# reflection, one edge diffraction (four wedge terms), one dual-number adjoint over (position, frequency, materials)
_REFLECT_FLOPS = 350
_DIFFRACT_FLOPS = 1200
_ADJOINT = 4.0
# mean paths per cell: reflection-type and diffraction, as the workloads have them
_CANYON_PATHS = (0.6, 15.0)
_TERRAIN_PATHS = (1.9, 0.0)
_CITY_PATHS = (3.0, 5.4)
# one cell of a map: receiver in; total power and field, four slots of power and field, diffraction vector, count out
_CELL_BYTES = 12 + 4 + 8 + 4 * (4 + 8) + 24 + 4


def _path_flops(cells, per_cell, components, depth, adjoint):
    refl = per_cell[0] * _REFLECT_FLOPS * (1 + depth) / 2.0
    diff = per_cell[1] * _DIFFRACT_FLOPS if "diffraction" in components else 0.0
    return cells * (refl + diff) * (1.0 + (_ADJOINT if adjoint else 0.0))


def work(case):
    kind = case["kind"]
    if kind == "two_ray":
        cells = case["rows"] * case["cols"]
        return {"bytes": cells * _CELL_BYTES, "flops": cells * (60 + _REFLECT_FLOPS)}
    if kind in ("map", "step"):
        cells = case["rows"] * case["cols"]
        adjoint = kind == "step" or case["ad"] != "none"
        return {"bytes": cells * _CELL_BYTES + 770 * 48 + 776 * 80,
                "flops": _path_flops(cells, _CANYON_PATHS, case["components"], case["depth"], adjoint)}
    if kind in ("points", "paths"):
        cells = int(_set_sizes(case).sum())
        scene = 776 * 48 + 776 * 80
        if kind == "points":
            return {"bytes": cells * _CELL_BYTES + scene,
                    "flops": _path_flops(cells, _CANYON_PATHS, case["components"], case["depth"], True)}
        rows = cells * sum(_CANYON_PATHS)
        row_bytes = 7 * 4 + 3 * 4 + case["depth"] * (4 + 4 + 12 + 12) + 8 + 8 + 24 + 12 + 12 + 16
        return {"bytes": cells * 28 + rows * row_bytes + scene,
                "flops": _path_flops(cells, _CANYON_PATHS, case["components"], case["depth"], False)}
    if kind == "terrain":
        cells = case["rows"] * case["cols"]
        return {"bytes": cells * _CELL_BYTES + 32738 * 48 + 16704 * 24,
                "flops": _path_flops(cells, _TERRAIN_PATHS, "los,reflection", case["depth"], True)}
    if kind == "city":
        t = case["tx"]
        sides = np.exp(np.linspace(math.log(case["side_min"]), math.log(case["side_max"]), t)) if t > 1 else \
            np.array([case["side_max"]])
        cells = 2 * int((np.round(sides) ** 2).sum())
        return {"bytes": cells * _CELL_BYTES + 134850 * 48,
                "flops": _path_flops(cells, _CITY_PATHS, case["components"], case["depth"], True)}
    if kind == "cfr":
        b, p, f = case["pairs"], case["paths"], case["subcarriers"]
        return {"bytes": b * p * 13 + b * f * 8, "flops": b * case["mean_paths"] * f * 14}
    if kind == "discover":
        pairs = case["sources"] * case["sinks"]
        rows = pairs * 1.5
        return {"bytes": (case["sources"] + case["sinks"]) * 40 + rows * (60 + 32 * case["depth"]),
                "flops": rows * _REFLECT_FLOPS * case["depth"]}
    if kind == "replay":
        rows = case["sources"] * case["sinks"] * case["slots"] * 0.5
        return {"bytes": rows * 2 * (60 + 32 * case["depth"]), "flops": rows * _REFLECT_FLOPS * case["depth"]}
    n, d = case["count"], case["depth"]
    row_in = 12 + 12 + 4 + 24 + d * (24 + 20)
    row_out = 24 + 8 + 8 + 4 + 4 + 4 + 12
    row_grad = 8 + 24 + d * (24 + 8)
    return {"bytes": n * (row_in + row_out + row_in + row_grad), "flops": n * d * _REFLECT_FLOPS * (1 + _ADJOINT)}


# ---------------------------------------------------------------- tolerance

def tolerance(case):
    """About four times what was measured: the two-ray map and the responses against ``exact`` (3.5e-7, 9e-7), row
    operators against ``exact`` (gradients with respect to materials and normals 6e-5: the slab's interior phase in
    float32), the canyon map's power against a 64-bit evaluation (5.6e-6), position gradients with the sums in
    another order (7e-7) on top of the maps' own difference."""
    kind = case["kind"]
    if kind in ("cfr", "two_ray"):
        return {"rel": 4.0e-6}
    if kind == "rows":
        return {"rel": 2.5e-4}
    if kind in ("paths", "discover", "replay") or case.get("ad") == "none":
        return {"rel": 2.0e-5}
    return {"rel": 3.0e-5}


# ---------------------------------------------------------------- exact

def exact(case, seed):
    if case["kind"] not in _EXACT:
        return None  # visibility of every candidate against every triangle: minutes on this box's host
    return _EXACT[case["kind"]](case, seed)


def _slab(cos_theta, eps, sigma, mu, gain, thickness, frequency):
    """Reflection of a slab in vacuum (TE, TM): interface coefficient with the interior bounces summed."""
    omega = 2.0 * math.pi * frequency
    eta = torch.complex(eps, -sigma / (omega * EPS0))
    ct = cos_theta.abs().clamp(1.0e-6, 1.0)
    root = torch.sqrt(eta * mu - (1.0 - ct * ct))
    te = (mu * ct - root) / (mu * ct + root)
    tm = (eta * ct - root) / (eta * ct + root)
    trip = torch.exp(-2.0j * (omega / C0) * thickness * root)
    return gain * te * (1.0 - trip) / (1.0 - te * te * trip), gain * tm * (1.0 - trip) / (1.0 - tm * tm * trip)


def _unit(v):
    return v / torch.linalg.vector_norm(v, dim=-1, keepdim=True)


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _transport(source, target, points, normals, tx_pol, eps, sigma, mu, gain, thickness, frequency):
    """Field vector at the target after the reflections at ``points`` [N, D, 3] (64-bit, differentiable)."""
    k = 2.0 * math.pi * frequency / C0
    prev = source
    outgoing = None
    value = None
    length = 0.0
    for b in range(points.shape[1]):
        seg = points[:, b] - prev
        length = length + torch.linalg.vector_norm(seg, dim=-1)
        direction = _unit(seg)
        if value is None:
            value = (tx_pol - direction * _dot(tx_pol, direction)).to(torch.complex128)
        n = _unit(normals[:, b])
        n = torch.where(_dot(direction, n) > 0, -n, n)
        cos_in = _dot(direction, n)
        outgoing = direction - 2.0 * cos_in * n
        s = _unit(torch.linalg.cross(n, direction))
        p_in = _unit(torch.linalg.cross(s, direction))
        p_out = _unit(torch.linalg.cross(s, outgoing))
        te, tm = _slab(cos_in[:, 0], eps[:, b], sigma[:, b], mu[:, b], gain[:, b], thickness[:, b], frequency)
        e_s, e_p = (value * s).sum(-1), (value * p_in).sum(-1)
        value = s * (te * e_s)[:, None] + p_out * (tm * e_p)[:, None]
        prev = points[:, b]
    seg = target - prev
    length = length + torch.linalg.vector_norm(seg, dim=-1)
    arrival = _unit(seg)
    carrier = torch.exp(-1.0j * (k * length)) / (2.0 * k * length)
    return value * carrier[:, None], arrival, length


def _exact_two_ray(case, seed):
    rows, cols = case["rows"], case["cols"]
    state = _prepare_two_ray(case, seed)
    f = case["frequency"]
    k = 2.0 * math.pi * f / C0
    d = dict(dtype=torch.float64)
    o = np.asarray(state.origin, np.float32)
    r = torch.as_tensor(o[0] + np.arange(rows, dtype=np.float32), **d)
    c = torch.as_tensor(o[1] + np.arange(cols, dtype=np.float32), **d)
    rx = torch.stack([r[:, None].expand(rows, cols), c[None, :].expand(rows, cols),
                      torch.full((rows, cols), float(o[2]), **d)], dim=-1).reshape(-1, 3)
    tx = torch.as_tensor(np.asarray(state.tx, np.float32), **d).expand_as(rx)
    pol = torch.tensor([0.0, 0.0, 1.0], **d).expand_as(rx)
    seg = rx - tx
    dist = torch.linalg.vector_norm(seg, dim=-1)
    u = _unit(seg)
    e = (pol - u * _dot(pol, u)) * (torch.exp(-1.0j * k * dist) / (2.0 * k * dist))[:, None]
    los = (e * (pol - u * _dot(pol, u))).sum(-1)
    t = tx[:, 2] / (tx[:, 2] + rx[:, 2])
    hit = torch.stack([tx[:, 0] + t * seg[:, 0], tx[:, 1] + t * seg[:, 1], torch.zeros_like(t)], dim=-1)
    one = torch.ones_like(t)[:, None]
    field, arrival, _ = _transport(tx, rx, hit[:, None], torch.tensor([0.0, 0.0, 1.0], **d).expand(len(t), 1, 3),
                                   pol, float(np.float32(5.31)) * one, float(np.float32(0.0326)) * one, one, one,
                                   5.0 * one, f)
    refl = (field * (pol - arrival * _dot(pol, arrival))).sum(-1)
    lay = lambda v: v.reshape(1, rows, cols).transpose(1, 2).contiguous()  # noqa: E731
    total = los + refl
    return {"path_gain": lay(total.abs() ** 2), "field": lay(total), "los": lay(los.abs() ** 2),
            "reflection": lay(refl.abs() ** 2), "los_field": lay(los), "reflection_field": lay(refl)}


def _exact_cfr(case, seed):
    s = _prepare_cfr(case, seed)
    tau = s.tau
    if s.normalize:
        low = torch.where(s.valid, tau, torch.full_like(tau, math.inf)).min(dim=1, keepdim=True).values
        tau = tau - low  # a float32 difference, as the response is defined
    tau = tau.to(torch.float64)
    freqs = s.freqs.to("cuda")
    out = torch.zeros((tau.shape[0], 1, freqs.numel()), dtype=torch.complex128, device="cuda")
    for p in range(tau.shape[1]):
        rows = torch.nonzero(s.valid[:, p]).flatten()
        for part in rows.split(16384):
            turns = tau[part, p, None] * freqs
            angle = -2.0 * math.pi * (turns - torch.floor(turns))
            out[part, 0] += s.a[part, p].to(torch.complex128) * torch.complex(torch.cos(angle), torch.sin(angle))
    return out


def _exact_rows(case, seed):
    s = _prepare_rows(case, seed)
    t = {k: v.detach().to(torch.float64) for k, v in s.t.items()}
    for k in _ROW_GRADS:
        t[k].requires_grad_(True)
    field, arrival, length = _transport(t["source"], t["target"], t["positions"], t["normals"], t["tx_pol"],
                                        t["eps"], t["sigma"], t["mu"], t["gain"], t["thickness"], s.frequency)
    perp = t["rx_pol"] - arrival * _dot(t["rx_pol"], arrival)
    coef = (field * perp).sum(-1)
    path_field = coef * torch.sqrt(t["power"])
    grads = torch.autograd.grad(path_field, [t[k] for k in _ROW_GRADS],
                                grad_outputs=s.weight.to(torch.complex128))
    out = {"field_vector": field, "coefficient": coef, "path_field": path_field, "path_gain": path_field.abs() ** 2,
           "path_length_m": length, "delay_s": length / C0, "direction": arrival}
    out = {k: v.detach() for k, v in out.items()}
    out.update({f"grad_{k}": g for k, g in zip(_ROW_GRADS, grads)})
    return out


_EXACT = {"two_ray": _exact_two_ray, "cfr": _exact_cfr, "rows": _exact_rows}
