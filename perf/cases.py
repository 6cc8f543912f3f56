"""The workloads whose speed this framework answers for.

`listed()` names twelve of them, `draw(rng)` gives others of the same ranges.
`prepare(case, seed)` builds what a program holds before its call (scene, rays,
partition, network), `run(state)` is one pass through the public entry points,
`work(case)` what a pass cannot do without, and `exact(case, seed)` the
floating-point outputs in 64 bits.

Hits, records, treelets and claim orders are exact by contract, so they are
returned as integer words (a hit record's floats by their bit patterns).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.abspath("treelet-prefetching-for-rt_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

HIT_WORDS, RECORD_WORDS = 20, 4
RECORDS_PER_RAY = 64  # room in the record buffer
TRIS_PER_INSTANCE = 1024  # 32 x 16 quads
STAGE_BYTES = 8192

# the network's layer widths (rtx_mlp): embedding, hidden, input row (169 used of 192)
EMB, HID, IN_PAD = 32, 128, 192
LEARNING_RATE = 1e-3
NO_TREELET = 0xFFFFFFFF


def listed():
    return [
        # one 32-lane warp of the simulated GPU: hits and the node-access trace
        # that traceRayWithTreelets hands the RT unit, called warp by warp
        dict(name="warp_treelet_records", op="trace", instances=0, width=8, height=4, bounce=0, order=1, records=1,
             budget=8192, stage=0),
        # the small scene the reference's CPU path runs: 16,384 camera rays, hits only
        dict(name="small_plain", op="trace", instances=0, width=128, height=128, bounce=0, order=0, records=0,
             budget=8192, stage=0),
        # the headline batch: 1M triangles, camera rays and one diffuse bounce per hit
        dict(name="diffuse_plain", op="trace", instances=1024, width=1024, height=1024, bounce=1, order=0, records=0,
             budget=8192, stage=0),
        # the same batch with every ray's node-access trace, in both visit orders:
        # what a caller replaying the accesses in a memory model asks for
        dict(name="diffuse_plain_records", op="trace", instances=1024, width=1024, height=1024, bounce=1, order=0,
             records=1, budget=8192, stage=0),
        dict(name="diffuse_treelet_records", op="trace", instances=1024, width=1024, height=1024, bounce=1, order=1,
             records=1, budget=8192, stage=0),
        # treelet order with the RT unit's prefetch heuristic staging whole treelets in LDS
        dict(name="diffuse_treelet_stage", op="trace", instances=1024, width=1024, height=1024, bounce=1, order=1,
             records=0, budget=8192, stage=1),
        # a 21M-triangle scene that no cache holds, treelet order, ragged image
        dict(name="large_treelet", op="trace", instances=20480, width=1919, height=1079, bounce=1, order=1, records=0,
             budget=8192, stage=0),
        # many scenes of very different sizes in one captured persistent launch
        dict(name="scenes_graph_plain", op="batch", scenes=16, max_tris=500_000, max_rays=524_288, order=0,
             budget=8192),
        # createTreelets on the 1M-triangle scene, the maps brought back as a simulator reads them
        dict(name="partition", op="partition", instances=1024, budget=8192),
        # the RT unit's ray-coherence schedule of an incoherent batch of a ragged size
        dict(name="coherence_order", op="order", instances=1024, width=1021, height=1013, bounce=1, hash="g"),
        # one epoch of the next-treelet network over the transitions of a traced
        # batch; the last batch is a short one
        dict(name="train_epoch", op="train", treelets=200_000, classes=16384, samples=65_700, batch=1024),
        # the network evaluated for the prefetch table's rows
        dict(name="predict_rows", op="predict", treelets=200_000, classes=16384, samples=20_011),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _image(rng, lo, hi):
    """A ragged image of about lo..hi pixels, wider than high."""
    n = _log_int(rng, lo, hi)
    h = max(1, int(math.sqrt(n / rng.uniform(1.0, 1.9))))
    return max(1, n // h), h


def draw(rng):
    op = rng.choice(["trace", "trace", "trace", "trace", "trace", "batch", "partition", "order", "train", "predict"])
    budget = rng.choice([1024, 2048, 4096, 8192, 16384])
    if op == "trace":
        instances = rng.choice([0, _log_int(rng, 3, 2048), _log_int(rng, 256, 8192)])
        w, h = _image(rng, 32, 1_100_000)
        stage = int(rng.random() < 0.15)
        return dict(op=op, instances=instances, width=w, height=h, bounce=rng.randrange(2), order=rng.randrange(2),
                    records=0 if stage else rng.randrange(2), budget=budget, stage=stage)
    if op == "batch":
        return dict(op=op, scenes=rng.randint(2, 16), max_tris=_log_int(rng, 10_000, 500_000),
                    max_rays=_log_int(rng, 16_384, 524_288), order=rng.randrange(2), budget=budget)
    if op == "partition":
        return dict(op=op, instances=_log_int(rng, 3, 1500), budget=budget)
    if op == "order":
        w, h = _image(rng, 4096, 1_100_000)
        return dict(op=op, instances=_log_int(rng, 16, 1024), width=w, height=h, bounce=rng.randrange(2),
                    hash=rng.choice("fgtd"))
    case = dict(op=op, treelets=_log_int(rng, 3000, 200_000), classes=_log_int(rng, 1000, 16384))
    if op == "train":
        return dict(case, samples=_log_int(rng, 3000, 65_700), batch=rng.choice([512, 1024, 2048]))
    return dict(case, samples=_log_int(rng, 500, 20_011))


# ---- inputs -------------------------------------------------------------------
class _Device:
    """A torch tensor as the device buffer the entry points take."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _words(n, width):
    return _Device(torch.zeros((n, width), dtype=torch.int32, device="cuda"))


def _upload(a):
    return _Device(torch.from_numpy(a.view(np.uint8).reshape(-1)).cuda())


def _scene_desc(rtx, instances, width, height, seed):
    if instances == 0:  # a displaced UV sphere of 16,384 triangles over a ground quad
        return rtx.workload_desc(rtx.WORKLOAD_SPHERE_AND_QUAD, slices=128, stacks=64, width=width, height=height,
                                 seed=seed, displacement=0.05)
    return rtx.workload_desc(rtx.WORKLOAD_INSTANCED_SPHERES, n_instances=instances, slices=32, stacks=16,
                             shared_blas=0, width=width, height=height, seed=seed,
                             box_size=max(4.0, 100.0 * (instances / 1024) ** (1 / 3)), scale_min=0.5, scale_max=2.0,
                             displacement=0.05)


def _bounce_rays(case):
    return case["width"] * case["height"] // 4 if case["bounce"] else 0


def _scene_and_rays(case, seed):
    """A context with the case's scene, its rays on the host and how many are camera rays."""
    import rtx

    ctx = rtx.Context(0)
    desc = _scene_desc(rtx, case["instances"], case["width"], case["height"], seed)
    scene = rtx.workload_scene(desc)
    ctx.set_scene(scene.arena, scene.tlas_offset)
    primary = rays = rtx.primary_rays(desc)
    n_bounce = _bounce_rays(case)
    if n_bounce:
        # one diffuse bounce at a hit, as many as a quarter of the pixels, evenly over the image
        bounce, _ = scene.secondary_rays(primary, ctx.trace(primary, mode=rtx.MODE_PLAIN), kind=0, seed=seed + 1)
        source = bounce if len(bounce) else primary
        rays = np.concatenate([primary, source[np.arange(n_bounce) * len(source) // n_bounce]])
    return ctx, rays, len(primary)


def _prepare_trace(case, seed):
    import rtx

    ctx, rays, n_primary = _scene_and_rays(case, seed)
    n = len(rays)
    options = dict(mode=rtx.MODE_TREELET if case["order"] else rtx.MODE_PLAIN)
    if case["order"] or case["stage"] or case["records"]:
        ctx.build_treelets(case["budget"])
    if case["stage"]:
        options.update(prefetch=rtx.PREFETCH_ALWAYS, stage_bytes=STAGE_BYTES)
    elif not case["order"] and n_primary < n:
        options["claim_start"] = n_primary  # the bounce rays first
    state = dict(ctx=ctx, n=n, rays=_upload(rays), hits=_words(n, HIT_WORDS), options=options)
    if case["records"]:
        state.update(offsets=_Device(torch.zeros(n + 1, dtype=torch.int64, device="cuda")),
                     records=_words(n * RECORDS_PER_RAY, RECORD_WORDS), capacity=n * RECORDS_PER_RAY)
    torch.cuda.synchronize()
    return state


def _prepare_batch(case, seed):
    import rtx
    from rtx import workloads

    # triangle and ray counts spread over the logarithm of their ranges; scenes and rays from the seed
    ctx = rtx.Context(0)
    k = case["scenes"]
    jobs = []
    for i in range(k):
        n = int(4096 * (case["max_rays"] / 4096) ** ((i + 0.5) / k))
        tris = 1000 * (case["max_tris"] / 1000) ** ((5 * i % k + 0.5) / k)
        width = int(math.ceil(math.sqrt(n / 2)))
        desc = workloads.scene_desc(tris, width, width, seed + 17 * i)
        scene = rtx.workload_scene(desc)
        ctx.set_scene(scene.arena, scene.tlas_offset)
        rays = workloads.mixed_rays(ctx, scene, desc, n, seed + i)
        sid = ctx.add_scene(scene.arena, scene.tlas_offset)
        if case["order"]:
            ctx.build_scene_treelets(sid, case["budget"])
        jobs.append((sid, _upload(rays), n, _words(n, HIT_WORDS)))
    torch.cuda.synchronize()
    # jobs are claimed in order: the longest first
    graph = ctx.batch_graph(jobs[::-1], mode=rtx.MODE_TREELET if case["order"] else rtx.MODE_PLAIN)
    return dict(ctx=ctx, graph=graph, jobs=jobs)


def _prepare_partition(case, seed):
    import rtx

    # One scene, its BLASes laid out in the seed's order: node offsets, and with
    # them every root, list and owner, differ, while their counts stay.
    rng, order = np.random.default_rng(2023), np.random.default_rng(seed)
    k = case["instances"]
    box = max(4.0, 100.0 * (k / 1024) ** (1 / 3))
    builder = rtx.SceneBuilder()
    blas = np.empty(k, np.int64)
    for i in order.permutation(k):
        blas[i] = builder.add_blas(rtx.displaced_sphere(32, 16, 1.0, 0.05, seed=1 + int(i)))
    for i in range(k):
        m = np.zeros((3, 4), np.float32)
        m[:, :3] = np.eye(3) * rng.uniform(0.5, 2.0)
        m[:, 3] = rng.uniform(0.0, box, 3)
        builder.add_instance(int(blas[i]), m, instance_id=i)
    scene = builder.finish()
    ctx = rtx.Context(0)
    ctx.set_scene(scene.arena, scene.tlas_offset)
    return dict(ctx=ctx, budget=case["budget"])


def _prepare_order(case, seed):
    ctx, rays, _ = _scene_and_rays(case, seed)
    n = len(rays)
    state = dict(ctx=ctx, n=n, rays=_upload(rays), hash=case["hash"], order=_words(n, 1), hashes=_words(n, 1))
    torch.cuda.synchronize()
    return state


def _parameter_shapes(case):
    t, c = case["treelets"], case["classes"]
    return [("E", (t + 1, EMB)), ("W1", (IN_PAD, HID)), ("b1", (HID,)), ("W2", (HID, HID)), ("b2", (HID,)),
            ("W3", (HID, EMB)), ("b3", (EMB,)), ("O", (c, EMB)), ("o", (c,))]


def _network(case, seed):
    """Parameters of a partly trained network (one FP32 vector, block by block) and samples
    of traced transitions: a few treelets are left far more often than the rest, their
    ancestors are shared, and the class entered follows from the treelet left."""
    rng = np.random.default_rng(seed)
    t, c, n = case["treelets"], case["classes"], case["samples"]
    spread = dict(E=0.5, W1=0.19, b1=0.02, W2=0.22, b2=0.02, W3=0.22, b3=0.02, O=0.3, o=0.05)
    parts = []
    for name, shape in _parameter_shapes(case):
        p = rng.uniform(-spread[name], spread[name], shape).astype(np.float32)
        if name == "W1":
            p[169:] = 0.0  # the padding of the input row
        parts.append(p.reshape(-1))
    cur = np.minimum((t * rng.random(n) ** 3).astype(np.int64), t - 1)
    level = 1 + (cur * 2654435761 % 17)
    hist = np.full((n, 4), NO_TREELET, np.int64)
    up = cur
    for k in range(4):
        up = up // 6
        hist[:, k] = np.where(level > k, up, NO_TREELET)
    target = (cur * 40503 + rng.integers(0, 4, n)) % c
    samples = dict(cur=cur, octant=rng.integers(0, 8, n), depth=(level / 32.0).astype(np.float32), hist=hist,
                   target=target)
    return np.concatenate(parts), samples


def _prepare_network(case, seed):
    import rtx

    params, columns = _network(case, seed)
    ctx = rtx.Context(0)
    net = ctx.mlp(case["treelets"], case["classes"])
    net.set_params(params)
    samples = np.zeros(case["samples"], rtx.MLP_SAMPLE_DTYPE)
    for name, column in columns.items():
        samples[name] = column
    return dict(ctx=ctx, net=net, samples=net.upload(samples), n=case["samples"], batch=case.get("batch"))


def prepare(case, seed):
    make = dict(trace=_prepare_trace, batch=_prepare_batch, partition=_prepare_partition, order=_prepare_order,
                train=_prepare_network, predict=_prepare_network)[case["op"]]
    return dict(make(case, seed), op=case["op"])


# ---- passes -------------------------------------------------------------------
def _check(status):
    if status != 0:
        import rtx

        raise rtx.RtxError(status, "pass")


def _run_trace(s):
    if "records" not in s:
        _check(s["ctx"].trace_device(s["rays"], s["n"], s["hits"], **s["options"]))
        return s["hits"].tensor
    _check(s["ctx"].trace_device(s["rays"], s["n"], s["hits"], records_buf=s["records"],
                                 record_capacity=s["capacity"], offsets_buf=s["offsets"], **s["options"]))
    return dict(hits=s["hits"].tensor, offsets=s["offsets"].tensor, records=s["records"].tensor)


def _run_batch(s):
    status, _ = s["graph"].launch(1)
    _check(status)
    return [hits.tensor for _, _, _, hits in s["jobs"]]


def _run_partition(s):
    summary = s["ctx"].build_treelets(s["budget"])
    t = s["ctx"].get_treelets()
    return dict(summary=summary, roots=t["roots"].view(np.int64), list_offsets=t["list_offsets"].view(np.int64),
                list_nodes=t["list_nodes"].view(np.int64), owner=t["owner"].view(np.int32))


def _run_order(s):
    import rtx

    _check(s["ctx"].coherence_order_device(s["rays"], s["n"], s["order"], hash=s["hash"],
                                           world=rtx.COHERENCE_WORLD_TLAS, hashes_buf=s["hashes"]))
    return dict(order=s["order"].tensor, hashes=s["hashes"].tensor)


def _run_train(s):
    loss = s["net"].train(s["samples"], n=s["n"], epochs=1, batch=s["batch"], lr=LEARNING_RATE)
    return dict(loss=loss, params=s["net"].params())


def _run_predict(s):
    top, prob = s["net"].predict(s["samples"], n=s["n"])
    return dict(top=top.view(np.int32), prob=prob)


_RUN = dict(trace=_run_trace, batch=_run_batch, partition=_run_partition, order=_run_order, train=_run_train,
            predict=_run_predict)


def run(state):
    return _RUN[state["op"]](state)


# ---- what a pass cannot do without ----------------------------------------------
def _arena_bytes(instances):
    """Nodes of the scene: about 88 bytes a triangle."""
    return 88 * (TRIS_PER_INSTANCE * instances if instances else 16386)


def work(case):
    op = case["op"]
    if op in ("trace", "order"):
        n = case["width"] * case["height"] + _bounce_rays(case)
    if op == "trace":
        # a ray visits about 17 nodes, tests six boxes of some 20 operations in each, and
        # records 21 accesses; the nodes are read once each, as far as the rays reach them
        read = min(_arena_bytes(case["instances"]), 17 * 64 * n)
        return dict(bytes=n * (64 + 80) + read + (n * (21 * 16 + 8) if case["records"] else 0),
                    flops=n * 17 * 6 * 20)
    if op == "batch":
        # the means of the spread counts
        rays = case["scenes"] * (case["max_rays"] - 4096) / math.log(case["max_rays"] / 4096)
        tris = case["scenes"] * (case["max_tris"] - 1000) / math.log(case["max_tris"] / 1000)
        return dict(bytes=rays * (64 + 80) + min(88 * tris, 12 * 64 * rays), flops=rays * 12 * 6 * 20)
    if op == "partition":
        # the arena read; an owner word and a list entry for each node
        arena = _arena_bytes(case["instances"])
        return dict(bytes=arena + arena / 64 * (4 + 8), flops=0)
    if op == "order":
        return dict(bytes=n * (64 + 4 + 4), flops=0)
    n, c = case["samples"], case["classes"]
    params = sum(math.prod(shape) for _, shape in _parameter_shapes(case))
    macs = n * (IN_PAD * HID + HID * HID + HID * EMB + EMB * c)
    if op == "train":
        # forward and backward; parameters and both Adam moments read and written
        return dict(bytes=n * 32 + params * 24, flops=6 * macs)
    return dict(bytes=n * (32 + 32) + params * 4, flops=2 * macs)


# ---- the network in 64 bits -------------------------------------------------------
def _exact_network(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    params, samples = _network(case, seed)
    flat = torch.from_numpy(params).to(device, torch.float64)
    samples = {k: torch.from_numpy(v).to(device) for k, v in samples.items()}
    return flat, samples


def _exact_logits(case, flat, samples, lo, hi):
    parts, at = {}, 0
    for name, shape in _parameter_shapes(case):
        size = math.prod(shape)
        parts[name] = flat[at:at + size].view(shape)
        at += size
    cur, hist = samples["cur"][lo:hi], samples["hist"][lo:hi]
    hist = torch.where(hist == NO_TREELET, case["treelets"], hist)
    one_hot = torch.nn.functional.one_hot(samples["octant"][lo:hi], 8).to(flat.dtype)
    x = torch.cat([parts["E"][cur], one_hot, samples["depth"][lo:hi, None].to(flat.dtype),
                   parts["E"][hist].reshape(hi - lo, 4 * EMB)], dim=1)
    h = torch.relu(x @ parts["W1"][:x.shape[1]] + parts["b1"])
    h = torch.relu(h @ parts["W2"] + parts["b2"])
    return (h @ parts["W3"] + parts["b3"]) @ parts["O"].T + parts["o"]


def _exact_train(case, seed):
    flat, samples = _exact_network(case, seed)
    m, v = torch.zeros_like(flat), torch.zeros_like(flat)
    total, steps = 0.0, 0
    for lo in range(0, case["samples"], case["batch"]):
        hi = min(case["samples"], lo + case["batch"])
        leaf = flat.detach().requires_grad_(True)
        loss = torch.nn.functional.cross_entropy(_exact_logits(case, leaf, samples, lo, hi), samples["target"][lo:hi])
        (g,) = torch.autograd.grad(loss, leaf)
        steps += 1
        total += float(loss.detach())
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        flat = flat - LEARNING_RATE * (m / (1 - 0.9 ** steps)) / (torch.sqrt(v / (1 - 0.999 ** steps)) + 1e-8)
    return dict(loss=total / steps, params=flat.cpu().numpy())


def _exact_predict(case, seed):
    flat, samples = _exact_network(case, seed)
    out = []
    for lo in range(0, case["samples"], 4096):
        hi = min(case["samples"], lo + 4096)
        out.append(torch.softmax(_exact_logits(case, flat, samples, lo, hi), dim=1).topk(4, dim=1).values)
    return dict(top=None, prob=torch.cat(out).cpu().numpy())


def exact(case, seed):
    """Only the network's outputs are rounded numbers; all others are exact words."""
    if case["op"] == "train":
        return _exact_train(case, seed)
    if case["op"] == "predict":
        return _exact_predict(case, seed)
    return None
