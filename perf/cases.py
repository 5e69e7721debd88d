"""Workloads of this framework as a program meets them, from the smallest call
to the largest: renders through each render entry point, ray queries, batches
of renders, the guiding network and vMF mixtures.

listed() gives the named workloads, draw(rng) one more of the same ranges;
prepare(case, seed) makes what a program holds before the call, run(state) is
one pass, work(case) its unavoidable bytes and operations, exact(case, seed)
the outputs in 64 bits where plain arithmetic gives them.
"""
import math

import numpy as np
import torch

from xitils_amd import api, scenes

_DEVICE = None


def _device():
    """The program's one device handle (its buffers are kept between calls)."""
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = api.Device(0)
    return _DEVICE


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # a thumbnail in a serving loop that must not allocate device memory: every material kind, one sample
        {"name": "thumbnail_96x64", "kind": "frame", "scene": "zoo", "entry": "static", "width": 96, "height": 64,
         "spp": 1, "depth": 8},
        # an interactive viewer: one sample per frame added to a host film, paths ended by roulette alone
        {"name": "viewer_800x800", "kind": "frame", "scene": "cornell", "entry": "host", "width": 800, "height": 800,
         "spp": 1, "depth": 0},
        # the Cornell box at its stated configuration
        {"name": "cornell_256x256x16", "kind": "frame", "scene": "cornell", "entry": "device", "width": 256,
         "height": 256, "spp": 16, "depth": 8},
        # a progressive 720p render of an indirectly lit room, four samples a call
        {"name": "room_720p_x4", "kind": "frame", "scene": "room", "triangles": 100000, "entry": "device",
         "width": 1280, "height": 720, "spp": 4, "depth": 16},
        # the same, its directions sampled from the guiding network as initialised (its first frames of training)
        {"name": "room_720p_x4_guided", "kind": "frame", "scene": "room", "triangles": 100000, "entry": "device",
         "width": 1280, "height": 720, "spp": 4, "depth": 16, "guided": True},
        # the headline: two million triangles under sun and sky, a whole 1080p frame
        {"name": "heightfield_1080p_x64", "kind": "frame", "scene": "heightfield", "cells": 1024, "entry": "device",
         "width": 1920, "height": 1080, "spp": 64, "depth": 16, "env_nee": True},
        # camera variants of a normal-mapped displaced plane under an image sky, in one call
        {"name": "plane_6_variants", "kind": "variants", "grid": 512, "variants": 6, "width": 960, "height": 540,
         "spp": 2, "depth": 12},
        # many small scenes in one call
        {"name": "rooms_16_x_128x128", "kind": "rooms", "rooms": 16, "side": 128, "spp": 4, "depth": 12,
         "most_triangles": 60000},
        # ray queries of another renderer: bounce rays of a 1080p frame, resident in device memory
        {"name": "rays_bounce_1080p", "kind": "rays", "query": "closest", "batch": "diffuse", "cells": 512,
         "width": 1920, "height": 1080, "on_device": True},
        # a few visibility probes from host arrays
        {"name": "rays_probe_1001", "kind": "rays", "query": "both", "batch": "diffuse", "cells": 64, "width": 143,
         "height": 7, "on_device": False},
        # directional samples of many texels fitted by vMF mixtures, mixtures evaluated and sampled
        {"name": "vmf_96_sets", "kind": "vmf", "sets": 96, "samples": 3000, "lobes": 6, "queries": 200000},
        # one step of training the guiding network on a program's own samples, with its gradient
        {"name": "guide_step_32768", "kind": "guide_step", "samples": 32768},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "variants", "rooms", "rays", "rays", "vmf", "guide_step"])
    if kind == "frame":
        scene = rng.choice(["cornell", "zoo", "room", "heightfield"])
        width = _log_int(rng, 48, 1920)
        height = max(16, int(width * rng.uniform(0.4, 1.1)))
        spp = _log_int(rng, 1, min(64, max(1, 60000000 // (width * height))))
        entry = rng.choice(["device", "device", "host", "static"])
        case = {"kind": kind, "scene": scene, "entry": entry, "width": width, "height": height, "spp": spp,
                "depth": rng.randint(2, 20)}
        if entry == "static":
            case["spp"] = max(1, min(spp, 4000000 // (width * height)))
        if entry != "static" and rng.random() < 0.2:
            case["depth"] = 0
        if scene == "heightfield":
            case["cells"] = _log_int(rng, 64, 1024)
            case["env_nee"] = rng.random() < 0.7
        if scene == "room":
            case["triangles"] = _log_int(rng, 5000, 200000)
            case["guided"] = entry != "static" and rng.random() < 0.5
        if not case.get("guided") and rng.random() < 0.2:
            case["naive"] = True
        return case
    if kind == "variants":
        return {"kind": kind, "grid": _log_int(rng, 64, 512), "variants": rng.randint(2, 8),
                "width": _log_int(rng, 128, 960), "height": _log_int(rng, 96, 540), "spp": rng.randint(1, 4),
                "depth": rng.randint(3, 12)}
    if kind == "rooms":
        return {"kind": kind, "rooms": rng.randint(3, 20), "side": rng.randint(64, 300), "spp": rng.randint(1, 8),
                "depth": rng.randint(4, 32), "most_triangles": 60000}
    if kind == "rays":
        return {"kind": kind, "query": rng.choice(["closest", "any", "both"]),
                "batch": rng.choice(["primary", "diffuse", "shadow"]), "cells": _log_int(rng, 64, 512),
                "width": _log_int(rng, 20, 1900), "height": _log_int(rng, 10, 1080), "on_device": rng.random() < 0.6}
    if kind == "vmf":
        return {"kind": kind, "sets": _log_int(rng, 4, 400), "samples": _log_int(rng, 50, 3000),
                "lobes": rng.randint(1, 12), "queries": _log_int(rng, 1000, 400000)}
    return {"kind": "guide_step", "samples": _log_int(rng, 500, 60000)}


# ---------------------------------------------------------------- prepare

def _frame_desc(case, seed):
    w, h = case["width"], case["height"]
    if case["scene"] == "heightfield":
        return scenes.heightfield(case["cells"], w, h, seed=2 + seed % 100003)
    if case["scene"] == "room":
        return scenes.occluded_room(w, h, n_tris=case["triangles"], seed=4 + seed % 100003)
    return scenes.material_zoo(w, h) if case["scene"] == "zoo" else scenes.cornell(w, h)


def _render_args(case, seed):
    args = {"seed": seed & 0x7FFFFFFF, "max_depth": case["depth"], "flags": 0}
    if case.get("env_nee"):
        args["flags"] |= api.XT_FLAG_ENV_NEE
    if case.get("guided"):
        args["flags"] |= api.XT_FLAG_GUIDE
    if case.get("naive"):
        args["integrator"] = 1
    return args


def _prepare_frame(case, seed):
    scene = api.Scene(_device(), _frame_desc(case, seed))
    if case.get("guided"):
        scene.guide_init(seed=1 + seed % 1000)
    state = {"case": case, "scene": scene, "args": _render_args(case, seed)}
    if case["entry"] == "host":   # a viewer's running sum
        state["film"] = np.zeros((case["height"], case["width"], 3), np.float32)
        state["done"] = 0
    else:
        state["film"] = torch.zeros((case["height"], case["width"], 3), dtype=torch.float32, device="cuda:0")
    return state


def _prepare_variants(case, seed):
    w, h = case["width"], case["height"]
    desc = scenes.displaced_plane(grid=case["grid"], width=w, height=h, normal_map_size=256, sky_size=(512, 256),
                                  seed=5 + seed % 100003)
    scene = api.Scene(_device(), desc)
    films = [torch.zeros((h, w, 3), dtype=torch.float32, device="cuda:0") for _ in range(case["variants"])]
    jobs = []
    for k, film in enumerate(films):
        kw = {"camera": scenes.displaced_plane_camera(k, w, h), "seed": seed & 0x7FFFFFFF, "max_depth": case["depth"],
              "flags": api.XT_FLAG_ENV_NEE}
        jobs.append((scene, w, h, case["spp"], (film.data_ptr(), False), kw))
    return {"case": case, "jobs": jobs, "films": films}


def _prepare_rooms(case, seed):
    master, jobs, films, index = 3 + seed % 100003, [], [], 0
    side = case["side"]
    while len(jobs) < case["rooms"]:
        first = np.random.default_rng([master, index]).uniform(math.log(1e4), math.log(2e6))
        if math.exp(first) <= case["most_triangles"]:   # the scene's triangle count is its first draw
            scene = api.Scene(_device(), scenes.batch_scene(index, master)[0])
            films.append(torch.zeros((side, side, 3), dtype=torch.float32, device="cuda:0"))
            jobs.append((scene, side, side, case["spp"], (films[-1].data_ptr(), False),
                         {"seed": (seed + index) & 0x7FFFFFFF, "max_depth": case["depth"]}))
        index += 1
    return {"case": case, "jobs": jobs, "films": films}


def _rays(case, seed):
    desc = scenes.heightfield(case["cells"], 1920, 1080, seed=2 + seed % 100003)
    return desc, scenes.ray_batch(desc, case["batch"], case["width"], case["height"], seed=seed % 100003)


def _prepare_rays(case, seed):
    desc, rays = _rays(case, seed)
    state = {"case": case, "scene": api.Scene(_device(), desc), "rays": rays}
    if case["on_device"]:
        n = rays.shape[0]
        state["rays"] = torch.from_numpy(rays).to("cuda:0")
        state["hits"] = torch.zeros((n, 4), dtype=torch.float32, device="cuda:0")
        state["occluded"] = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    return state


def _unit(v):
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _vmf_inputs(case, seed):
    """Mixtures (the library's encoding), samples drawn from them, the fit's
    start uniforms, and the evaluation's and the sampler's inputs."""
    rng = np.random.default_rng([seed, 11])
    sets, n, lobes, q = case["sets"], case["samples"], case["lobes"], case["queries"]
    mu = _unit(rng.normal(size=(sets, lobes, 3)))
    kappa = np.exp(rng.uniform(math.log(3.0), math.log(120.0), (sets, lobes)))
    alpha = rng.dirichlet(np.full(lobes, 4.0), sets)
    pick = (rng.random((sets, n, 1)) > np.cumsum(alpha, axis=1)[:, None, :-1]).sum(axis=2)
    at = np.arange(sets)[:, None]
    m, k = mu[at, pick], kappa[at, pick]
    u, phi = rng.random((sets, n)), rng.uniform(0, 2 * math.pi, (sets, n))
    w = np.clip(1.0 + np.log(u + (1.0 - u) * np.exp(-2.0 * k)) / k, -1.0, 1.0)
    t = _unit(np.cross(m, np.where(np.abs(m[..., :1]) < 0.9, [1.0, 0.0, 0.0], [0.0, 1.0, 0.0])))
    b = np.cross(m, t)
    r = np.sqrt(1.0 - w * w)
    x = w[..., None] * m + (r * np.cos(phi))[..., None] * t + (r * np.sin(phi))[..., None] * b
    enc = np.concatenate([mu, kappa[..., None], alpha[..., None]], axis=2).reshape(sets, 5 * lobes)[:, :-1]
    return {"mixtures": np.ascontiguousarray(enc, np.float32), "samples": x.reshape(-1, 3).astype(np.float32),
            "offsets": (np.arange(sets + 1) * n).astype(np.uint32),
            "init": rng.random((sets, 2 * lobes)).astype(np.float32),
            "dirs": _unit(rng.normal(size=(q, 3))).astype(np.float32),
            "uniforms": rng.random((q, 4)).astype(np.float32),
            "which": rng.integers(0, sets, q).astype(np.uint32)}


def _guide_inputs(case, seed):
    """A network's parameters (the flat layout of xitils_amd.h) and weighted
    direction samples at points of the unit cube."""
    rng = np.random.default_rng([seed, 12])
    n = case["samples"]
    params = np.zeros(api.GUIDE_NUM_PARAMS, np.float32)
    at = 0
    for rows, cols, used, scale in ((64, 96, 64, 1.0), (64, 64, 64, 1.0), (64, 64, 64, 1.0), (48, 64, 40, 0.3)):
        bound = scale * math.sqrt(6.0 / cols)
        params[at:at + used * cols] = rng.uniform(-bound, bound, used * cols)
        params[at + rows * cols:at + rows * cols + used] = rng.uniform(-0.05, 0.05, used)
        at += rows * cols + rows
    normal = _unit(rng.normal(size=(n, 3)))
    wo = _unit(normal + 0.9 * _unit(rng.normal(size=(n, 3))))
    target = _unit(np.array([0.5, 0.999, 0.5]) + 0.1 * rng.normal(size=(n, 3)) * [1, 0, 1] - (p := rng.random((n, 3))))
    spread = _unit(normal + _unit(rng.normal(size=(n, 3))))
    dirs = np.where(rng.random((n, 1)) < 0.5, target, spread)
    return {"params": params, "queries": np.concatenate([p, normal, wo], axis=1).astype(np.float32),
            "dirs": dirs.astype(np.float32), "weights": rng.exponential(1.0, n).astype(np.float32)}


def prepare(case, seed):
    if case["kind"] == "frame":
        return _prepare_frame(case, seed)
    if case["kind"] == "variants":
        return _prepare_variants(case, seed)
    if case["kind"] == "rooms":
        return _prepare_rooms(case, seed)
    if case["kind"] == "rays":
        return _prepare_rays(case, seed)
    if case["kind"] == "vmf":
        return {"case": case, **_vmf_inputs(case, seed)}
    state = {"case": case, "scene": api.Scene(_device(), scenes.cornell(64, 64)), **_guide_inputs(case, seed)}
    state["scene"].guide_init()
    state["scene"].guide_set_params(state["params"])
    return state


# ---------------------------------------------------------------- run

def _clear(films):
    """Zeroed device films: the library renders on its own streams, so their
    clearing is waited for."""
    for film in films:
        film.zero_()
    torch.cuda.current_stream().synchronize()


def _run_frame(state):
    case, scene, film = state["case"], state["scene"], state["film"]
    size = (case["width"], case["height"], case["spp"])
    if case["entry"] == "host":
        scene.render(*size, film=film, spp_offset=state["done"], **state["args"])
        state["done"] += case["spp"]
        return film
    _clear([film])
    render = scene.render_static if case["entry"] == "static" else scene.render_device
    render(film.data_ptr(), *size, **state["args"])
    return film


def _hits(hits):
    prim = hits[:, 1].contiguous().view(torch.int32) if isinstance(hits, torch.Tensor) else hits[:, 1].copy().view(np.int32)
    return {"t": hits[:, 0], "prim": prim, "b": hits[:, 2:4]}


def _run_rays(state):
    scene, rays, query, out = state["scene"], state["rays"], state["case"]["query"], {}
    if state["case"]["on_device"]:
        n = rays.shape[0]
        if query != "any":
            scene.trace_closest_dev(rays.data_ptr(), n, state["hits"].data_ptr())
            out.update(_hits(state["hits"]))
        if query != "closest":
            scene.trace_any_dev(rays.data_ptr(), n, state["occluded"].data_ptr())
            out["occluded"] = state["occluded"]
        return out
    if query != "any":
        out.update(_hits(scene.trace_closest(rays)))
    if query != "closest":
        out["occluded"] = scene.trace_any(rays)
    return out


def run(state):
    kind = state["case"]["kind"]
    if kind == "frame":
        return _run_frame(state)
    if kind in ("variants", "rooms"):
        _clear(state["films"])
        api.render_batch(state["jobs"])
        return state["films"]
    if kind == "rays":
        return _run_rays(state)
    if kind == "vmf":
        dev = _device()
        fit, steps = api.vmf_fit(dev, state["case"]["lobes"], state["samples"], state["offsets"], state["init"])
        return {"fit": fit, "steps": steps,
                "pdf": api.vmf_eval(dev, state["mixtures"], state["dirs"], state["which"]),
                "sampled": api.vmf_sample(dev, state["mixtures"], state["uniforms"], state["which"])}
    scene = state["scene"]
    gradient = scene.guide_gradient(state["queries"], state["dirs"], state["weights"])
    scene.guide_train_step(state["queries"], state["dirs"], state["weights"])
    return {"gradient": gradient, "params": scene.guide_params()}


# ---------------------------------------------------------------- work

_NODE, _TRI = 64, 48             # bytes of a BVH node and of a triangle
_VISIT, _TEST = 60, 60           # operations of a node's four boxes and of a triangle's test
_SHADE = 400                     # operations of a vertex: random numbers, BSDF sample and evaluation, light sample


def _ray_flops(triangles):
    return (2.0 + 0.8 * math.log2(triangles + 4.0)) * _VISIT * 0.7 + 3.0 * _TEST


def _path_work(triangles, width, height, spp, rays_per_path):
    paths = width * height * spp
    scene = triangles * (_TRI + 0.25 * _NODE)
    touched = min(scene, paths * rays_per_path * (2.0 * _NODE + _TRI))   # a small frame reads only a part of a large scene
    return {"bytes": touched + 24.0 * width * height,
            "flops": paths * rays_per_path * (_ray_flops(triangles) + 0.5 * _SHADE)}


def _scene_triangles(case):
    return {"cornell": 36, "zoo": 1000, "room": case.get("triangles", 0), "heightfield": 2 * case.get("cells", 0) ** 2}[case["scene"]]


def work(case):
    if case["kind"] == "frame":
        # vertices that a path visits, with a shadow ray at most of them: open scenes let paths out early
        rays = 2.6 if case["scene"] == "heightfield" else 1.6 * min(case["depth"] or 12, 12) + 1.0
        w = _path_work(_scene_triangles(case), case["width"], case["height"], case["spp"], rays)
        if case.get("guided"):
            w["flops"] += case["width"] * case["height"] * case["spp"] * 0.6 * rays * 33792.0
        return w
    if case["kind"] == "variants":
        one = _path_work(2 * case["grid"] ** 2, case["width"], case["height"], case["spp"], 3.0)
        return {"bytes": one["bytes"] + (case["variants"] - 1) * 24.0 * case["width"] * case["height"],
                "flops": case["variants"] * one["flops"]}
    if case["kind"] == "rooms":
        one = _path_work(25000, case["side"], case["side"], case["spp"], 1.2 * min(case["depth"], 8))
        return {"bytes": case["rooms"] * one["bytes"], "flops": case["rooms"] * one["flops"]}
    if case["kind"] == "rays":
        n, triangles = case["width"] * case["height"], 2 * case["cells"] ** 2
        passes = 2 if case["query"] == "both" else 1
        out = {"closest": 16, "any": 1, "both": 17}[case["query"]]
        touched = min(triangles * (_TRI + 0.25 * _NODE), n * (2.0 * _NODE + _TRI))
        return {"bytes": n * (32.0 + out) + touched, "flops": passes * n * _ray_flops(triangles)}
    if case["kind"] == "vmf":
        sets, n, lobes, q = case["sets"], case["samples"], case["lobes"], case["queries"]
        data = sets * (12.0 * n + 4 * (5 * lobes - 1) * 2 + 8 * lobes) + q * (12 + 4 + 4 + 16 + 4 + 12)
        return {"bytes": data, "flops": 40.0 * sets * n * lobes * 30 + 40.0 * q * lobes}   # some 20 operations of a pdf, and its sums; tens of EM steps
    n = case["samples"]
    return {"bytes": 52.0 * n + 6 * 4.0 * api.GUIDE_NUM_PARAMS, "flops": 2.0 * n * 89088.0}


# ---------------------------------------------------------------- exact

def _exact_vmf(case, seed):
    """pdf and samples of the mixtures, from the closed forms."""
    x = _vmf_inputs(case, seed)
    lobes = case["lobes"]
    e = np.concatenate([x["mixtures"].astype(np.float64), np.zeros((case["sets"], 1))], axis=1).reshape(-1, lobes, 5)
    e[:, -1, 4] = 1.0 - e[:, :-1, 4].sum(axis=1)
    m, k, a = e[x["which"], :, :3], e[x["which"], :, 3], e[x["which"], :, 4]
    d = x["dirs"].astype(np.float64)
    cosine = np.einsum("qlc,qc->ql", m, d)
    pdf = (a * k / (2 * math.pi * (1 - np.exp(-2 * k))) * np.exp(k * (cosine - 1))).sum(axis=1)
    return {"fit": None, "steps": None, "pdf": pdf, "sampled": None}


def _features(q):
    p, cols = q[:, :3].clamp(0.0, 1.0), []
    for axis in range(3):
        for band in range(12):
            angle = math.pi * p[:, axis] * 2.0 ** band
            cols += [torch.sin(angle), torch.cos(angle)]
    return torch.cat([torch.stack(cols, 1), q[:, 3:], torch.zeros(q.shape[0], 18, dtype=q.dtype)], 1)


def _exact_guide(case, seed):
    """Gradient of the sum of -w log q(dir | query) by autograd in 64 bits."""
    x = _guide_inputs(case, seed)
    flat = torch.from_numpy(x["params"].astype(np.float64)).requires_grad_(True)
    q, d, w = (torch.from_numpy(x[k].astype(np.float64)) for k in ("queries", "dirs", "weights"))
    h, at = _features(q), 0
    for layer, (rows, cols) in enumerate(((64, 96), (64, 64), (64, 64), (48, 64))):
        h = h @ flat[at:at + rows * cols].reshape(rows, cols).T + flat[at + rows * cols:at + rows * cols + rows]
        at += rows * cols + rows
        if layer < 3:
            h = torch.relu(h)
    y = h[:, :40].reshape(-1, 8, 5)
    mu = y[..., :3] / y[..., :3].norm(dim=2, keepdim=True)
    k = torch.exp(y[..., 3].clamp(-3.0, 9.0))
    log_lobe = torch.log(k / (2 * math.pi * (1 - torch.exp(-2 * k)))) + k * ((mu * d[:, None]).sum(2) - 1)
    (-(w * torch.logsumexp(torch.log_softmax(y[..., 4], 1) + log_lobe, 1)).sum()).backward()
    return {"gradient": flat.grad.numpy(), "params": None}


def _exact_probes(case, seed):
    """Closest distances by testing every triangle (Moeller-Trumbore)."""
    desc, rays = _rays(case, seed)
    o, d = (torch.from_numpy(rays[:, s].astype(np.float64)).to("cuda:0") for s in (slice(0, 3), slice(4, 7)))
    v = torch.from_numpy(desc.objects[0].positions[desc.objects[0].indices].astype(np.float64)).to("cuda:0")
    e1, e2, best = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0], []
    for a in range(0, o.shape[0], 128):
        oo, dd = o[a:a + 128, None], d[a:a + 128, None]
        p = torch.linalg.cross(dd, e2[None])
        det = (p * e1).sum(2)
        s = oo - v[None, :, 0]
        b1 = (s * p).sum(2) / det
        r = torch.linalg.cross(s, e1[None].expand_as(s))
        b2 = (r * dd).sum(2) / det
        t = (r * e2).sum(2) / det
        ok = (det != 0) & (b1 >= 0) & (b2 >= 0) & (b1 + b2 <= 1) & (t > 0)
        best.append(torch.where(ok, t, math.inf).min(1).values)
    return {"t": torch.cat(best), "prim": None, "b": None, "occluded": None}


def exact(case, seed):
    if case["kind"] == "vmf":
        return _exact_vmf(case, seed)
    if case["kind"] == "guide_step":
        return _exact_guide(case, seed)
    if case["kind"] == "rays" and case["query"] != "any" and case["width"] * case["height"] * case["cells"] ** 2 <= 100_000_000:
        return _exact_probes(case, seed)
    # a film is a sum over random paths, whose branches follow the rounding of
    # every step before them: it has no value of its own in 64 bits
    return None
