"""Performance cases of the NeuS / Neuralangelo training-and-render path.

Each case is one pass through the package's public entry points at a size and
form that the workloads of `bench.py` and the reference's configurations meet:

  field       VolumeSDF.forward and its backward to every parameter, the body
              of a training step (central differences or the analytic
              gradient, with or without the curvature evaluations)
  radiance    VolumeRadiance / VolumeDualColor forward and backward
  background  VolumeDensity (unbounded-sphere contraction, stand-alone hash
              grid and MLP) forward and backward
  step        a whole training call: NeuSModel.forward on given samples, the
              loss terms and the gradients of every parameter
  query       SDF, gradient and feature of scattered points, no backward
  lattice     the marching-cubes SDF lattice (`sdf_grid`)
  render      an eval-mode NeuSModel.forward: march, field, colour, composite

`exact` restates each path in float64 with plain torch (GPU or CPU).
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "instant-angelo_amd"))

FINE_SCALE = 1.3195079107728942     # 16 levels from 32 to 2049
# the grid and SDF network of the workloads: (levels, base, scale, hidden
# layers, outputs)
SPHERE = dict(levels=8, base=16, scale=1.5, hidden=1, out=16)
NEURALANGELO = dict(levels=16, base=32, scale=FINE_SCALE, hidden=1, out=16)
CONFIG = dict(levels=16, base=32, scale=FINE_SCALE, hidden=2, out=65)


def listed():
    return [
        # a probe of a few points (surface projection, picking): launches and
        # latency alone
        dict(name="query-1k", kind="query", n=1001, rows=19, active=16, **NEURALANGELO),
        # the marching-cubes lattice of a validation export, 64^3-point chunks
        dict(name="lattice-128", kind="lattice", resolution=128, rows=21, active=16,
             **NEURALANGELO),
        # the plain NeuS step's field: 1024 rays x 64 samples, 8 levels
        dict(name="field-sphere", kind="field", n=65536, rows=15, active=8, grad="fd",
             curvature=True, precision="fp32", **SPHERE),
        # one step's field at the reference's initial 256 rays (ragged, odd)
        dict(name="field-256-rays", kind="field", n=20011, rows=19, active=16, grad="fd",
             curvature=True, precision="fp32", **NEURALANGELO),
        # the flagship step's field: 8192 rays, 2^21 rows a level
        dict(name="field-8192-rays", kind="field", n=940000, rows=21, active=16, grad="fd",
             curvature=True, precision="fp32", **NEURALANGELO),
        # the same in the mixed-precision form, half the rays
        dict(name="field-mixed", kind="field", n=470003, rows=21, active=16, grad="fd",
             curvature=True, precision="mixed", **NEURALANGELO),
        # the start of training: the progressive band at 4 levels
        dict(name="field-band-4", kind="field", n=480000, rows=19, active=4, grad="fd",
             curvature=True, precision="fp32", **NEURALANGELO),
        # the reference's own configuration: analytic gradients, 65 outputs
        dict(name="field-analytic", kind="field", n=490000, rows=19, active=16,
             grad="analytic", curvature=True, precision="fp32", **CONFIG),
        # its texture (68 features + 16 SH + normal, dual colour)
        dict(name="radiance-dual", kind="radiance", n=490000, features=68, dual=True,
             precision="fp32"),
        # the learned background's field at one step's samples
        dict(name="background", kind="background", n=230000, rows=19, active=16),
        # a whole training call: forward, losses, gradients of 2048 rays' samples
        dict(name="step", kind="step", n=240007, rows=19, active=16, grad="fd",
             precision="fp32", **NEURALANGELO),
        # a 128 x 128 novel view in chunks of 2048 rays
        dict(name="render-128", kind="render", n=16384, rows=19, active=16, **NEURALANGELO),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["field", "field", "field", "radiance", "background", "step", "query",
                       "lattice", "render"])
    rows = rng.choice([19, 20, 21])
    if kind == "field":
        form = rng.choice([SPHERE, NEURALANGELO, NEURALANGELO, CONFIG])
        active = form["levels"] if rng.random() < 0.7 else rng.randint(4, form["levels"])
        grad = "analytic" if form is CONFIG or rng.random() < 0.15 else "fd"
        return dict(kind=kind, n=_spread(rng, 1000, 700000),
                    rows=15 if form is SPHERE else rows, active=active, grad=grad,
                    curvature=rng.random() < 0.8,
                    precision="mixed" if rng.random() < 0.25 else "fp32", **form)
    if kind == "radiance":
        wide = rng.random() < 0.5
        return dict(kind=kind, n=_spread(rng, 1000, 900000), features=68 if wide else 19,
                    dual=wide, precision="mixed" if rng.random() < 0.25 else "fp32")
    if kind == "background":
        return dict(kind=kind, n=_spread(rng, 1000, 400000), rows=19, active=rng.randint(4, 16))
    if kind == "step":
        return dict(kind=kind, n=_spread(rng, 5000, 500000), rows=rows, active=16,
                    grad=rng.choice(["fd", "analytic"]), precision="fp32", **NEURALANGELO)
    if kind == "query":
        return dict(kind=kind, n=_spread(rng, 100, 500000), rows=rows, active=16,
                    **rng.choice([NEURALANGELO, CONFIG]))
    if kind == "lattice":
        return dict(kind=kind, resolution=_spread(rng, 24, 200), rows=rows, active=16,
                    **NEURALANGELO)
    return dict(kind=kind, n=_spread(rng, 500, 25000), rows=rows, active=16, **NEURALANGELO)


# ---- inputs (plain torch, from the seed alone) ----------------------------
def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=gen.device)


def _rand(gen, *shape):
    return torch.rand(*shape, generator=gen, device=gen.device)


def _levels(case):
    """tcnn's level table: (scale, resolution, first row, rows, hashed)."""
    out, offset = [], 0
    log2 = np.float32(math.log2(float(np.float32(case["scale"]))))
    for level in range(case["levels"]):
        p = np.float32(2.0 ** float(np.float32(level) * log2))
        scale = np.float32(p * np.float32(case["base"])) - np.float32(1.0)
        res = int(math.ceil(float(scale))) + 1
        rows = min((res ** 3 + 7) // 8 * 8, 1 << case["rows"])
        out.append((float(scale), res, offset, rows, res ** 3 > rows))
        offset += rows
    return out, offset


def _sdf_scene(p):
    s = (p - p.new_tensor([0.25, 0.0, 0.0])).norm(dim=-1) - 0.35
    q = p - p.new_tensor([-0.2, 0.0, 0.1])
    ring = torch.stack([q[..., :2].norm(dim=-1) - 0.45, q[..., 2]], -1).norm(dim=-1) - 0.12
    return torch.minimum(s, ring)


STEP = 2.0 / 1024


def _rays(gen, n):
    eye = F.normalize(_randn(gen, n, 3), dim=-1) * 2.5
    aim = F.normalize(_randn(gen, n, 3), dim=-1) * (_rand(gen, n, 1) ** (1 / 3)) * 0.55
    return torch.cat([eye, F.normalize(aim - eye, dim=-1)], -1)


def _marched(gen, n):
    """n samples in ray order as an occupancy-pruned march leaves them: steps
    of 2/1024 where the scene's SDF is below 0.02 (a band and the inside).
    Returns rays, ray_indices, t_starts, t_ends, packed."""
    k = torch.arange(1024, device=gen.device)
    rays, counts, t_all = [], [], []
    left = n
    while left > 0:
        r = _rays(gen, min(max(left // 96, 16), 4096))
        t0 = 1.5 + _rand(gen, r.shape[0], 1) * STEP + k * STEP
        pos = r[:, None, :3] + r[:, None, 3:] * (t0 + 0.5 * STEP)[..., None]
        keep = _sdf_scene(pos) < 0.02
        c = keep.sum(1)
        done = torch.cumsum(c, 0)
        c = torch.where(done > left, (left - (done - c)).clamp(min=0), c)
        t_all.append(t0[keep][:min(left, int(done[-1]))])
        rays.append(r)
        counts.append(c)
        left -= int(c.sum())
    rays, counts = torch.cat(rays).contiguous(), torch.cat(counts)
    t0 = torch.cat(t_all).contiguous()
    ridx = torch.repeat_interleave(torch.arange(rays.shape[0], device=gen.device), counts)
    packed = torch.stack([torch.cumsum(counts, 0) - counts, counts], -1).int().contiguous()
    return rays, ridx.int(), t0, t0 + STEP, packed


def _points(gen, n):
    rays, ridx, t0, t1, _ = _marched(gen, n)
    i = ridx.long()
    return (rays[i, :3] + rays[i, 3:] * ((t0 + t1) * 0.5)[:, None]).contiguous(), rays[i, 3:]


def _table(gen, case, size):
    """Trained-like rows: each level adds detail of its own cell size."""
    levels, total = _levels(case)
    t = _randn(gen, total, 2)
    for _, res, offset, rows, _ in levels:
        t[offset:offset + rows] *= size * 32.0 / res
    return t


def _layers(gen, dims, weight_norm, sdf=False):
    """(v, g, bias) per layer (g None without weight norm)."""
    out = []
    for i, (a, b) in enumerate(zip(dims[:-1], dims[1:])):
        v = _randn(gen, b, a) * math.sqrt(2.0 / (b if sdf else a))
        bias = _randn(gen, b) * 0.05
        if sdf and i == 0:
            v[:, 3:] *= 0.6
        if sdf and i == len(dims) - 2:
            v = _randn(gen, b, a) / 8
            v[0] = math.sqrt(math.pi) / 8 + 1e-3 * v[0]
            bias[0] = -0.5
        g = v.norm(dim=1, keepdim=True) * (1 + 0.02 * _randn(gen, b, 1)) if weight_norm else None
        out.append((v, g, bias))
    return out


def _sdf_inputs(gen, case):
    dims = [3 + 2 * case["levels"]] + [64] * case["hidden"] + [case["out"]]
    return dict(table=_table(gen, case, 0.02), mlp=_layers(gen, dims, True, sdf=True))


def _inputs(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    I = {}
    if kind in ("field", "query", "lattice", "render", "step"):
        I.update(_sdf_inputs(gen, case))
    if kind == "field":
        n = case["n"]
        I["pts"], _ = _points(gen, n)
        I["randn"] = _randn(gen, n, 3)
        # upstream gradients at the scale of mean losses (10 rgb, 0.1 eikonal,
        # 0.5 curvature), times the loss scale in the mixed form
        u = (65536.0 if case["precision"] == "mixed" else 1.0) / n
        I["up"] = [_randn(gen, n) * u, _randn(gen, n, 3) * (0.2 * u),
                   _randn(gen, n, case["out"] + 3) * u]
        if case["curvature"]:
            I["up"].append(0.5 * u * _rand(gen, n, 1))
    elif kind == "query":
        I["pts"], _ = _points(gen, case["n"])
    elif kind == "radiance":
        n, f = case["n"], case["features"]
        _, dirs = _points(gen, n)
        I["dirs"] = dirs.contiguous()
        I["feature"] = _randn(gen, n, f) * 0.5
        I["normal"] = F.normalize(_randn(gen, n, 3), dim=-1)
        I["mlp"] = _layers(gen, [f + 19, 64, 64, 3], False)
        I["up"] = _randn(gen, n, 3) * ((65536.0 if case["precision"] == "mixed" else 1.0) / n)
    elif kind == "background":
        n = case["n"]
        r = _rays(gen, n // 128 + 1)
        i = torch.arange(n, device=gen.device) // 128
        t = 1.5 * torch.exp((torch.arange(n, device=gen.device) % 128 + _rand(gen, n)) * 0.05)
        I["pts"] = (r[i, :3] + r[i, 3:] * (2.0 + t)[:, None]).contiguous()
        I["table"] = _table(gen, _background_grid(case), 0.5)
        I["mlp"] = _layers(gen, [35, 64, 8], False)
        I["up"] = [_randn(gen, n) / n, _randn(gen, n, 8) / n]
    elif kind == "render":
        n = case["n"]
        side = math.ceil(math.sqrt(n))
        eye = F.normalize(_randn(gen, 3), dim=0) * 2.5
        fwd = -eye / eye.norm()
        right = F.normalize(torch.linalg.cross(fwd, _randn(gen, 3)), dim=0)
        up = torch.linalg.cross(right, fwd)
        k = torch.arange(n, device=gen.device)
        x, y = ((k % side) + 0.5) / side - 0.5, (k // side + 0.5) / side - 0.5
        d = F.normalize(fwd + 0.73 * (x[:, None] * right - y[:, None] * up), dim=-1)
        I["rays"] = torch.cat([eye.expand(n, 3), d], -1).contiguous()
    if kind == "step":
        n = case["n"]
        I["rays"], *samples = _marched(gen, n)
        I["samples"] = tuple(samples)
        I["randn"] = _randn(gen, n, 3)
        I["rgb"] = _rand(gen, I["rays"].shape[0], 3)
    if kind in ("step", "render"):
        I["rad"] = _layers(gen, [case["out"] + 22, 64, 64, 3], False)
    return I


def _background_grid(case):
    return dict(levels=16, base=32, scale=FINE_SCALE, rows=case["rows"])


# ---- what a user's program holds ------------------------------------------
def _band(case, levels, base, scale):
    return {"otype": "ProgressiveBandHashGrid", "n_levels": levels, "n_features_per_level": 2,
            "log2_hashmap_size": case["rows"], "base_resolution": base, "per_level_scale": scale,
            "include_xyz": True, "start_level": case["active"], "start_step": 1 << 30,
            "update_steps": 1000}


def _mlp(hidden, **kw):
    return dict({"otype": "VanillaMLP", "activation": "ReLU", "output_activation": "none",
                 "n_neurons": 64, "n_hidden_layers": hidden}, **kw)


def _geometry_config(case):
    return {"name": "volume-sdf", "radius": 1.0, "feature_dim": case["out"],
            "grad_type": "analytic" if case.get("grad") == "analytic" else "finite_difference",
            "finite_difference_eps": "progressive", "isosurface": None,
            "precision": case.get("precision", "fp32"),
            "xyz_encoding_config": _band(case, case["levels"], case["base"], case["scale"]),
            "mlp_network_config": _mlp(case["hidden"], sphere_init=True, sphere_init_radius=0.5,
                                       weight_norm=True)}


def _texture_config(features, dual, precision):
    return {"name": "volume-dual-color" if dual else "volume-radiance",
            "input_feature_dim": features + 3, "precision": precision,
            "dir_encoding_config": {"otype": "SphericalHarmonics", "degree": 4},
            "mlp_network_config": _mlp(2), "color_activation": "sigmoid"}


@torch.no_grad()
def _fill(network, layers):
    for lin, (v, g, b) in zip(network.linears(), layers):
        (lin.weight if g is None else lin.weight_v).copy_(v)
        if g is not None:
            lin.weight_g.copy_(g)
        lin.bias.copy_(b)


def _leaves(network):
    out = []
    for lin in network.linears():
        out += [lin.weight_v, lin.weight_g] if hasattr(lin, "weight_g") else [lin.weight]
        out.append(lin.bias)
    return out


@torch.no_grad()
def _fill_grid(grid, table):
    grid.params.copy_(table.reshape(-1))


def prepare(case, seed):
    from angelo_amd import make
    from angelo_amd.system import NeuSTrainer
    from angelo_amd.utils import to_config
    I = _inputs(case, seed)
    kind, dev = case["kind"], torch.device("cuda:0")
    S = dict(case=case, I=I)
    if kind in ("field", "query", "lattice"):
        geo = make("volume-sdf", to_config(_geometry_config(case))).to(dev)
        _fill(geo.network, I["mlp"])
        _fill_grid(geo.grid_module, I["table"])
        geo.train(kind == "field")
        geo.update_step(0, 0)
        S["model"] = geo
        S["params"] = [geo.grid_module.params] + _leaves(geo.network)
    elif kind == "radiance":
        tex = make("volume-dual-color" if case["dual"] else "volume-radiance",
                   to_config(_texture_config(case["features"], case["dual"],
                                             case["precision"]))).to(dev)
        _fill(tex.network, I["mlp"])
        S["model"] = tex
        S["params"] = [I["feature"].requires_grad_(), I["normal"].requires_grad_()] \
            + _leaves(tex.network)
    elif kind == "background":
        bg = make("volume-density", to_config({
            "name": "volume-density", "radius": 1.0, "feature_dim": 8,
            "density_activation": "trunc_exp", "density_bias": -1, "isosurface": None,
            "xyz_encoding_config": _band(case, 16, 32, FINE_SCALE),
            "mlp_network_config": _mlp(1)})).to(dev)
        net = bg.encoding_with_network
        grid = net.encoding.encoding.encoding
        _fill(net.network, I["mlp"])
        _fill_grid(grid, I["table"])
        S["model"], S["params"] = bg, [grid.params] + _leaves(net.network)
    else:
        render = kind == "render"
        cfg = to_config({
            "name": "neus", "radius": 1.0, "num_samples_per_ray": 512, "train_num_rays": 256,
            "max_train_num_rays": 8192, "ray_chunk": 2048, "randomized": True,
            "grid_prune": render, "grid_prune_occ_thre": 0.001, "cos_anneal_end": 20000,
            "learned_background": False, "background_color": "white",
            "render_step_size": STEP, "max_samples_per_ray": 512,
            "precision": case.get("precision", "fp32"),
            "variance": {"init_val": 0.3, "modulate": False},
            "geometry": _geometry_config(case),
            "texture": _texture_config(case["out"] + 3, False, case.get("precision", "fp32"))})
        model = make("neus", cfg).to(dev)
        _fill(model.geometry.network, I["mlp"])
        _fill(model.texture.network, I["rad"])
        _fill_grid(model.geometry.grid_module, I["table"])
        model.train(not render)
        model.update_step(0, 20001)
        S["model"] = model
        S["params"] = ([model.geometry.grid_module.params] + _leaves(model.geometry.network)
                       + _leaves(model.texture.network) + [model.variance.variance])
        if render:
            c = (torch.arange(128, device=dev) + 0.5) / 64 - 1.0
            p = torch.stack(torch.meshgrid(c, c, c, indexing="ij"), -1)
            model.occupancy_grid.binary.copy_((_sdf_scene(p) < 0.02).to(torch.uint8))
        else:
            sys_cfg = to_config({"loss": {"lambda_rgb_mse": 10.0, "lambda_eikonal": 0.1,
                                          "lambda_curvature": 0.5}})
            S["trainer"] = NeuSTrainer(model, sys_cfg, cfg)
            S["trainer"].global_step = 20001
    return S


def run(S):
    case, I, m = S["case"], S["I"], S["model"]
    kind = case["kind"]
    if kind == "lattice":
        return m.sdf_grid(case["resolution"])
    if kind == "query":
        return m(I["pts"], with_grad=True, with_feature=True)
    if kind == "render":
        with torch.no_grad():
            out = m(I["rays"])
        return [out[k] for k in ("comp_rgb_full", "opacity", "depth", "comp_normal",
                                 "num_samples")]
    if kind == "field":
        outs = m(I["pts"], with_grad=True, with_feature=True, with_laplace=case["curvature"],
                 randn=I["randn"])
        return list(outs) + list(torch.autograd.grad(outs, S["params"], I["up"]))
    if kind == "radiance":
        rgb = m(I["feature"], I["dirs"], I["normal"])
        return [rgb] + list(torch.autograd.grad(rgb, S["params"], I["up"]))
    if kind == "background":
        outs = m(I["pts"])
        return list(outs) + list(torch.autograd.grad(outs, S["params"], I["up"]))
    out = m(I["rays"], samples=I["samples"], randn=I["randn"])
    loss, _ = S["trainer"].losses(out, {"rgb": I["rgb"]})
    return ([loss] + [out[k] for k in ("comp_rgb_full", "opacity", "depth")]
            + list(torch.autograd.grad(loss, S["params"])))


# ---- what a pass cannot do without ----------------------------------------
def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "radiance":
        w = (case["features"] + 19) * 64 + 64 * 64 + 64 * 3
        cols = case["features"] + 3
        return {"bytes": 4.0 * n * (2 * cols + 3 + 6) + 8.0 * w, "flops": 6.0 * n * w}
    if kind == "background":
        table = 8.0 * _levels(_background_grid(case))[1]
        w = 35 * 64 + 64 * 8
        touched = min(table, 64.0 * n * case["active"])
        return {"bytes": touched + table + 4.0 * n * (3 + 9 + 9),
                "flops": n * (6.0 * w + 2 * case["active"] * 8 * 4)}
    table = 8.0 * _levels(case)[1]
    w = (3 + 2 * case["levels"]) * 64 + 64 * 64 * (case["hidden"] - 1) + 64.0
    wide = w + 64.0 * (case["out"] - 1)
    encode = case["active"] * 8 * 4.0
    if kind == "lattice":
        n = case["resolution"] ** 3
        return {"bytes": min(table, 64.0 * n * case["active"]) + 4.0 * n,
                "flops": n * (2 * w + encode)}
    if kind == "render":
        n = 60 * n     # samples of a ray that the scene's grid keeps, about
    fd = case.get("grad", "fd") == "fd"
    evals = 1 + (6 if fd else 0) + (6 if case.get("curvature", kind == "step") else 0)
    flops = n * (2 * wide + (evals - 1) * 2 * w + evals * encode)
    if case.get("precision") == "mixed":
        table *= 0.75   # fp16 rows read, fp32 gradient written
    touched = min(table, 64.0 * n * evals * case["active"])
    if kind == "query":
        return {"bytes": touched + 4.0 * n * (3 + 4 + case["out"] + 3), "flops": flops}
    rad = (case["out"] + 22) * 64 + 64 * 64 + 64 * 3
    if kind == "render":
        return {"bytes": touched + case["n"] * 4.0 * 14, "flops": flops + 2.0 * n * rad}
    if kind == "field":
        return {"bytes": touched + table + 4.0 * n * (6 + 2 * (case["out"] + 8)),
                "flops": 3 * flops}
    return {"bytes": touched + table + 4.0 * n * 6, "flops": 3 * flops + 6.0 * n * rad}


# ---- float64 --------------------------------------------------------------
class _Grid64:
    """Hash-grid encode in float64; `taps` collects (rows, gathered values)
    so that the table's gradient can be added up after a backward."""

    def __init__(self, case, table, active):
        self.levels, _ = _levels(case)
        self.table = table.double()
        self.active = active
        self.taps = []

    def __call__(self, x, grad):
        feats = []
        for k, (scale, res, offset, rows, hashed) in enumerate(self.levels):
            if k >= self.active:
                feats.append(x.new_zeros(x.shape[0], 2))
                continue
            pos = x * scale + 0.5
            cell = torch.floor(pos.detach())
            f = pos - cell
            c = cell.long()
            bit = torch.tensor([[b & 1, b >> 1 & 1, b >> 2] for b in range(8)], device=x.device)
            v = c[:, None, :] + bit
            if hashed:
                idx = v[..., 0] ^ (v[..., 1] * 2654435761 & 0xFFFFFFFF) \
                    ^ (v[..., 2] * 805459861 & 0xFFFFFFFF)
            else:
                idx = v[..., 0] + v[..., 1] * res + v[..., 2] * res * res
            idx = offset + idx % rows
            w = torch.where(bit.bool(), f[:, None, :], 1 - f[:, None, :]).prod(-1)
            val = self.table[idx]
            if grad:
                val.requires_grad_(True)
                self.taps.append((idx, val))
            feats.append((w[..., None] * val).sum(1))
        return torch.cat(feats, -1)

    def collect(self, out):
        for idx, val in self.taps:
            if val.grad is not None:
                out.index_add_(0, idx.reshape(-1), val.grad.reshape(-1, 2))
        self.taps = []


class _Mlp64:
    def __init__(self, layers, act):
        self.leaves = [[t.double().requires_grad_(True) for t in lay if t is not None]
                       for lay in layers]
        self.act = act

    def __call__(self, h):
        for i, lay in enumerate(self.leaves):
            w = lay[0] if len(lay) == 2 else \
                lay[0] * (lay[1] / lay[0].norm(dim=1, keepdim=True))
            h = h @ w.t() + lay[-1]
            if i < len(self.leaves) - 1:
                h = self.act(h)
        return h

    def grads(self):
        return [t.grad if t.grad is not None else torch.zeros_like(t)
                for lay in self.leaves for t in lay]


def _softplus(h):
    return F.softplus(h, beta=100)


class _Field64:
    """VolumeSDF in float64 (radius 1): sdf, grad, normal, feature, laplace."""

    def __init__(self, case, I):
        self.case = case
        self.grid = _Grid64(case, I["table"].half() if case.get("precision") == "mixed"
                            else I["table"], case["active"])
        self.mlp = _Mlp64(I["mlp"], _softplus)
        self.eps = 2.0 / (case["base"] * case["scale"] ** (case["active"] - 1))

    def net(self, x01, grad):
        return self.mlp(torch.cat([x01 * 2 - 1, self.grid(x01, grad)], -1))

    def central(self, base, grad):
        step = torch.eye(3, device=base.device, dtype=base.dtype) * self.eps
        p = torch.stack([base + s * step[d] for d in range(3) for s in (1, -1)])
        x = (p.clamp(-1, 1) + 1) / 2
        s = self.net(x.reshape(-1, 3), grad)[:, 0].reshape(6, -1)
        return torch.stack([(s[2 * d] - s[2 * d + 1]) / (2 * self.eps) for d in range(3)], -1)

    def __call__(self, pts, randn, curvature, with_grad=True, grad=False):
        p = pts.double()
        x0 = (p + 1) / 2
        analytic = with_grad and self.case.get("grad") == "analytic"
        if analytic:
            x0.requires_grad_(True)
        with torch.set_grad_enabled(grad or analytic):
            out = self.net(x0, grad)
            r = dict(sdf=out[:, 0], feature=torch.cat([out, x0 * 2 - 1], -1))
            if not with_grad:
                return r
            if analytic:
                g, = torch.autograd.grad(out[:, 0].sum(), x0, create_graph=grad)
                r["grad"] = g / 2
            else:
                r["grad"] = self.central(p, grad)
            r["normal"] = F.normalize(r["grad"], dim=-1)
            if curvature:
                t = torch.linalg.cross(r["normal"], F.normalize(randn.double(), dim=-1))
                n2 = F.normalize(self.central(x0.detach() + t * self.eps, grad), dim=-1)
                dot = (r["normal"] * n2).sum(-1).clamp(-1 + 1e-6, 1 - 1e-6)
                r["laplace"] = (torch.acos(dot) / math.pi)[:, None]
        return r


CHUNK = 1 << 15


def _field_all(field, pts, randn, curvature, with_grad=True):
    parts = []
    for a in range(0, pts.shape[0], CHUNK):
        r = field(pts[a:a + CHUNK], randn[a:a + CHUNK] if randn is not None else None, curvature,
                  with_grad)
        parts.append({k: v.detach() for k, v in r.items()})
    return {k: torch.cat([q[k] for q in parts]) for k in parts[0]}


def _field_backward(field, pts, randn, curvature, up):
    """Gradients [table, layers...] for upstream gradients by output name."""
    g_table = torch.zeros_like(field.grid.table)
    for a in range(0, pts.shape[0], CHUNK):
        s = slice(a, a + CHUNK)
        r = field(pts[s], randn[s], curvature, grad=True)
        torch.autograd.backward([r[k] for k in up], [u[s].double() for u in up.values()])
        field.grid.collect(g_table)
    return [g_table.reshape(-1)] + field.mlp.grads()


def _sh16(d):
    x, y, z = d.unbind(-1)
    xx, yy, zz = x * x, y * y, z * z
    pi = math.pi
    c1 = math.sqrt(3 / (4 * pi))
    c2 = math.sqrt(15 / pi)
    c3 = math.sqrt(35 / (2 * pi)) / 4
    c4 = math.sqrt(21 / (2 * pi)) / 4
    return torch.stack([
        torch.full_like(x, 0.5 / math.sqrt(pi)), -c1 * y, c1 * z, -c1 * x, c2 / 2 * x * y,
        -c2 / 2 * y * z, math.sqrt(5 / pi) / 4 * (3 * zz - 1), -c2 / 2 * x * z,
        c2 / 4 * (xx - yy), -c3 * y * (3 * xx - yy), math.sqrt(105 / pi) / 2 * x * y * z,
        -c4 * y * (5 * zz - 1), math.sqrt(7 / pi) / 4 * z * (5 * zz - 3),
        -c4 * x * (5 * zz - 1), math.sqrt(105 / pi) / 4 * z * (xx - yy),
        -c3 * x * (xx - 3 * yy)], -1)


def _radiance64(mlp, feature, dirs, normal, dual):
    rgb = torch.sigmoid(mlp(torch.cat([feature, _sh16(dirs), normal], -1)))
    return rgb + torch.sigmoid(feature[:, 1:4]) if dual else rgb


def _exact_background(case, I):
    grid = _Grid64(_background_grid(case), I["table"], case["active"])
    mlp = _Mlp64(I["mlp"], torch.relu)
    x = I["pts"].double()
    mag = x.norm(dim=-1, keepdim=True)
    m = torch.where(mag > 1, mag, torch.ones_like(mag))
    x = torch.where(mag > 1, (2 - 1 / m) * (x / m), x) / 4 + 0.5
    out = mlp(torch.cat([x * 2 - 1, grid(x, True)], -1))
    density = torch.exp(out[:, 0] - 1)
    torch.autograd.backward([density, out], [u.double() for u in I["up"]])
    g = torch.zeros_like(grid.table)
    grid.collect(g)
    return [density.detach(), out.detach(), g.reshape(-1)] + mlp.grads()


def _exact_step(case, I):
    field = _Field64(case, I)
    rad = _Mlp64(I["rad"], torch.relu)
    ridx, t0, t1, packed = I["samples"]
    rays, i = I["rays"].double(), ridx.long()
    t0, t1 = t0.double(), t1.double()
    mid, dist = (t0 + t1) / 2, t1 - t0
    dirs = rays[i, 3:]
    pts = rays[i, :3] + dirs * mid[:, None]
    f = _field_all(field, pts, I["randn"], True)
    names = ("sdf", "grad", "normal", "feature", "laplace")
    leaf = {k: f[k].clone().requires_grad_(True) for k in names}
    variance = torch.tensor(0.3, dtype=torch.float64, device=pts.device, requires_grad=True)
    inv_s = torch.exp(variance * 10)
    rgb = _radiance64(rad, leaf["feature"], dirs, leaf["normal"], False)
    cos = -F.relu(-(dirs * leaf["normal"]).sum(-1))
    nxt = torch.sigmoid((leaf["sdf"] + cos * dist * 0.5) * inv_s)
    prv = torch.sigmoid((leaf["sdf"] - cos * dist * 0.5) * inv_s)
    alpha = ((prv - nxt + 1e-5) / (prv + 1e-5)).clip(0, 1)
    R, most = rays.shape[0], int(packed[:, 1].max())
    at = torch.arange(i.shape[0], device=i.device) - packed[:, 0].long()[i]
    through = torch.ones(R, most + 1, dtype=alpha.dtype, device=alpha.device)
    through = torch.cumprod(through.index_put((i, at + 1), 1 - alpha), 1)
    w = through[i, at] * alpha
    add = lambda v: torch.zeros(R, v.shape[1], dtype=v.dtype, device=v.device).index_add(0, i, v)
    opacity, depth, crgb = add(w[:, None]), add((w * mid)[:, None]), add(w[:, None] * rgb)
    full = crgb + (1 - opacity)
    ok = opacity[:, 0] > 0
    loss = 10 * F.mse_loss(full[ok], I["rgb"].double()[ok]) \
        + 0.1 * ((leaf["grad"].norm(dim=-1) - 1) ** 2).mean() + 0.5 * leaf["laplace"].abs().mean()
    loss.backward()
    up = {k: leaf[k].grad for k in names if leaf[k].grad is not None}
    g = _field_backward(field, pts, I["randn"], True, up)
    return [loss.detach(), full.detach(), opacity.detach(), depth.detach()] + g + rad.grads() \
        + [variance.grad]


def exact(case, seed):
    kind = case["kind"]
    if kind == "render":
        return None      # the marched sample positions are a chain of fp32 steps
    I = _inputs(case, seed)
    if kind == "lattice":
        a = torch.arange(-1.0, 1.0, 2.0 / case["resolution"]).to(_device())
        pts = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
        sdf = _field_all(_Field64(case, I), pts, None, False, with_grad=False)["sdf"]
        return sdf.view(len(a), len(a), len(a))
    if kind == "query":
        f = _field_all(_Field64(case, I), I["pts"], None, False)
        return [f["sdf"], f["grad"], f["feature"]]
    if kind == "field":
        field = _Field64(case, I)
        f = _field_all(field, I["pts"], I["randn"], case["curvature"])
        names = ["sdf", "grad", "feature"] + (["laplace"] if case["curvature"] else [])
        g = _field_backward(field, I["pts"], I["randn"], case["curvature"],
                            dict(zip(names, I["up"])))
        return [f[k] for k in names] + g
    if kind == "radiance":
        mlp = _Mlp64(I["mlp"], torch.relu)
        feature, normal = (I[k].double().requires_grad_(True) for k in ("feature", "normal"))
        rgb = _radiance64(mlp, feature, I["dirs"].double(), normal, case["dual"])
        rgb.backward(I["up"].double())
        return [rgb.detach(), feature.grad, normal.grad] + mlp.grads()
    if kind == "background":
        return _exact_background(case, I)
    return _exact_step(case, I)
