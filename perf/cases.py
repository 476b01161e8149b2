"""Work that users of the encoding have it do, as measurable cases.

A case is one geometry of the encoding (input dimension, levels, features, capacity), one batch of
points and one use of it through ``PermutoEncoding``, autograd and the package's optimizers:

  infer     the encoding of a batch under ``no_grad``: rendering, meshing, sphere tracing
  train     forward, then backward w.r.t. the table from the gradient the layer after the encoding hands back
  step      ``train`` with ``zero_grad`` before it and the optimizer's step on the table after it
  eikonal   forward, gradient w.r.t. the positions with ``create_graph``, backward of a loss on that gradient
  sdf       ``eikonal`` with a loss on the encoded values themselves in the same backward (an SDF training step)
  sdf_step  ``sdf`` with the optimizer's step on the table

``draw`` gives more of the same over the ranges: 2 to 8 dimensions, 6 to 24 levels, 2, 4 or 8
features, 2^12 to 2^22 slots per level (powers of two and not), 200 to 2^20 points, unordered, near a
surface or along rays, a table gathered in 32 or 16 bits, all levels on or a coarse-to-fine window.
"""
import math

import numpy as np
import torch

import permutohedral_encoding_amd as pe
from permutohedral_encoding_amd.optim import AdamW, SparseTableAdamW

RAY_SAMPLES = 128
TABLES = {"fp32": False, "fp16": torch.float16, "bf16": torch.bfloat16}


def _case(**given):
    case = {"use": "infer", "pos_dim": 3, "levels": 24, "features": 2, "capacity": 1 << 18, "points": 1 << 20,
            "order": "uniform",    # "uniform" in the unit cube, "sphere" (near a surface) or "rays" (samples along rays, in order)
            "finest": 1e-4,        # scales are geomspace(1, finest, levels)
            "window_t": 1.0,       # position in the coarse-to-fine schedule; 1: no window is passed
            "table": "fp32",       # what the kernels gather from
            "concat_points": False, "contiguous_output": False, "sparse_table_grad": False, "skip_zero_gradients": False}
    assert set(given) <= set(case) | {"name"}
    case.update(given)
    return case


def listed():
    return [
        # the last rays of a sphere tracer, a few probes of a field: what one call costs
        _case(name="infer_1k", points=1000),
        # a chunk of a rendered image or of a marching-cubes grid
        _case(name="infer_64k", points=1 << 16),
        # rendering from a large trained table, gathered in 16 bits
        _case(name="infer_bf16_2e22", points=500_003, capacity=1 << 22, order="sphere", table="bf16"),
        # a training step on a small batch with a small table: a toy SDF, an interactive fit
        _case(name="step_4k", use="step", points=4097, levels=16, capacity=1 << 16, finest=1e-3),
        # an image or a plane fitted with four features per level
        _case(name="step_d2_f4", use="step", points=1 << 18, pos_dim=2, levels=16, features=4, capacity=1 << 16, finest=1e-3),
        # the headline configuration: 2^20 unordered points, table gradient
        _case(name="train_1m", use="train"),
        # a renderer's training batch: samples along rays, points concatenated, dense rows, levels still easing in
        _case(name="train_rays", use="train", points=131_007, order="rays", window_t=0.7, concat_points=True, contiguous_output=True),
        # high-dimensional scaling
        _case(name="train_d8", use="train", points=1 << 19, pos_dim=8, levels=16, capacity=1 << 19, finest=1e-3),
        # an SDF training step on the batch of a few hundred rays
        _case(name="sdf_32k", use="sdf", points=1 << 15, order="sphere"),
        # space-time field: gradient of the gradient w.r.t. the positions
        _case(name="eikonal_d4_1m", use="eikonal", pos_dim=4),
        # an SDF training step on a table that no cache holds, fine levels masked
        _case(name="sdf_1m_2e22", use="sdf", capacity=1 << 22, order="sphere", window_t=16 / 24),
        # the same table, an ordinary batch, gradient and optimizer following what the batch touches
        _case(name="sdf_step_sparse_2e22", use="sdf_step", points=200_001, capacity=1 << 22, order="sphere", window_t=16 / 24,
              sparse_table_grad=True),
    ]


def _cost(case):
    """Rough cost: table accesses of all passes, and the values of the dense arrays that are walked."""
    passes = {"infer": 1, "train": 3, "step": 3, "eikonal": 6, "sdf": 9, "sdf_step": 9}[case["use"]]
    accesses = case["points"] * case["levels"] * (case["pos_dim"] + 1) * case["features"] // 2
    return passes * accesses, case["levels"] * case["capacity"] * case["features"]


def draw(rng):
    most = [max(c) for c in zip(*(_cost(c) for c in listed()))]
    while True:
        use = rng.choice(["infer", "infer", "train", "train", "step", "eikonal", "sdf", "sdf_step"])
        log2_points = rng.uniform(math.log2(200), 20)
        points = int(2 ** log2_points)
        if rng.random() < 0.25:
            points = 1 << round(log2_points)
        log2_capacity = rng.uniform(12, 22)
        capacity = int(2 ** log2_capacity) if rng.random() < 0.2 else 1 << round(log2_capacity)
        case = _case(use=use, points=points, capacity=capacity,
                     pos_dim=rng.choice([2, 3, 3, 3, 4, 4, 5, 6, 7, 8]), levels=rng.randint(6, 24),
                     features=rng.choice([2, 2, 2, 4, 8]), order=rng.choice(["uniform", "sphere", "rays"]),
                     finest=rng.choice([1e-4, 1e-3, 1e-2]), concat_points=rng.random() < 0.25,
                     contiguous_output=rng.random() < 0.25, skip_zero_gradients=rng.random() < 0.5)
        if rng.random() < 0.4:
            case["window_t"] = round(rng.uniform(0.3, 1.0), 3)
        if use in ("infer", "train"):
            case["table"] = rng.choice(["fp32", "fp32", "fp16", "bf16"])
        if use == "sdf_step" or (use == "step" and rng.random() < 0.3):
            case["sparse_table_grad"] = rng.random() < 0.5
        # nothing dearer than the dearest listed case
        if all(a <= b for a, b in zip(_cost(case), most)):
            return case


def _positions(case, generator):
    n, d = case["points"], case["pos_dim"]
    kw = dict(generator=generator, device="cuda")
    if case["order"] == "uniform":
        return torch.rand((n, d), **kw)
    if case["order"] == "sphere":
        u = torch.randn((n, d), **kw)
        return 0.5 + (0.5 + 0.02 * torch.randn((n, 1), **kw)) * u / u.norm(dim=1, keepdim=True)
    rays = -(-n // RAY_SAMPLES)
    origin = 0.25 + 0.5 * torch.rand((rays, 1, d), **kw)
    direction = torch.randn((rays, 1, d), **kw)
    direction = direction / direction.norm(dim=2, keepdim=True)
    along = (torch.arange(RAY_SAMPLES, device="cuda") + torch.rand((rays, RAY_SAMPLES), **kw)) / RAY_SAMPLES - 0.5
    return (origin + 0.8 * along[:, :, None] * direction).clamp(0.0, 1.0).reshape(-1, d)[:n].contiguous()


def prepare(case, seed):
    """The encoding with a trained-looking table, its optimizer, the points, and the gradients the layers after it hand back."""
    torch.manual_seed(seed)
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    scales = np.geomspace(1.0, case["finest"], num=case["levels"])
    with torch.device("cuda"):
        enc = pe.PermutoEncoding(case["pos_dim"], case["capacity"], case["levels"], case["features"], scales,
                                 concat_points=case["concat_points"], lattice_half_precision=TABLES[case["table"]],
                                 sparse_table_grad=case["sparse_table_grad"], contiguous_output=case["contiguous_output"])
    with torch.no_grad():
        enc.lattice_values.mul_(1e4)
    n, rows = case["points"], (case["points"], enc.output_dims())
    kw = dict(generator=generator, device="cuda")
    state = {"use": case["use"], "enc": enc, "positions": _positions(case, generator),
             "schedule": pe.Coarse2Fine(case["levels"]) if case["window_t"] < 1.0 else None, "t": case["window_t"], "optimizer": None}
    if case["use"] == "infer":
        enc.eval()
        return state
    # gradients of a loss that is a mean over the points
    state["grad_encoded"] = torch.randn(rows, **kw) / n
    if case["use"] in ("eikonal", "sdf", "sdf_step"):
        state["positions"].requires_grad_(True)
        state["grad_value"] = torch.randn(rows, **kw).requires_grad_(True)  # d(network output)/d(encoded): depends on the network's weights
        state["grad_normal"] = torch.randn((n, case["pos_dim"]), **kw) / n
    if case["use"] in ("step", "sdf_step"):
        options = dict(lr=1e-3, betas=(0.9, 0.99), weight_decay=0.0)
        if case["sparse_table_grad"]:
            state["optimizer"] = SparseTableAdamW(enc, **options)
        else:
            state["optimizer"] = AdamW([enc.lattice_values], skip_zero_gradients=case["skip_zero_gradients"], **options)
    return state


def run(state):
    enc, positions = state["enc"], state["positions"]
    window = state["schedule"](state["t"]) if state["schedule"] is not None else None
    if state["use"] == "infer":
        with torch.no_grad():
            return enc(positions, window)
    optimizer = state["optimizer"]
    if optimizer is not None:
        optimizer.zero_grad()
    else:
        enc.lattice_values.grad = None
    encoded = enc(positions, window)
    out = {"encoded": encoded}
    if state["use"] in ("train", "step"):
        encoded.backward(state["grad_encoded"])
    else:
        positions.grad = state["grad_value"].grad = None
        normal, = torch.autograd.grad(encoded, positions, state["grad_value"], create_graph=True)
        if state["use"] == "eikonal":
            normal.backward(state["grad_normal"])
        else:
            torch.autograd.backward([encoded, normal], [state["grad_encoded"], state["grad_normal"]])
            out["positions_grad"] = positions.grad
        out["normal"], out["grad_value_grad"] = normal, state["grad_value"].grad
    if optimizer is not None:
        optimizer.step()
        out["table"] = enc.lattice_values
    else:
        out["table_grad"] = enc.lattice_values.grad
    return out


def work(case):
    """Bytes: positions, gradients and results once per use that needs them; of the table the slots a batch can touch,
    of a dense table gradient and of a dense optimizer step every entry.  Operations: the simplex search and the sums."""
    n, d, f, use = case["points"], case["pos_dim"], case["features"], case["use"]
    levels = min(case["levels"], math.ceil(case["levels"] * case["window_t"]))
    extra = math.ceil(d / f) if case["concat_points"] else 0
    columns = f * (case["levels"] + extra)
    table = case["levels"] * case["capacity"] * f
    touched = levels * min(case["capacity"], n * (d + 1)) * f
    value_bytes = 4 if case["table"] == "fp32" else 2
    nbytes = 4 * n * d + value_bytes * touched + 4 * n * columns
    passes = 1
    if use != "infer":
        nbytes += 4 * n * columns + (4 * touched if case["sparse_table_grad"] else 4 * table)
        passes = 2
    if use in ("eikonal", "sdf", "sdf_step"):
        nbytes += 4 * n * (columns + 2 * d) + (4 * n * (columns + d) if use != "eikonal" else 0)
        passes = 4 if use == "eikonal" else 6
    if use in ("step", "sdf_step"):
        nbytes += 4 * 6 * (touched if case["sparse_table_grad"] or case["skip_zero_gradients"] else table)
    flops = passes * n * levels * ((d + 1) * (d + 1) + 12 * (d + 1) + 2 * f * (d + 1))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # 32-bit sums in any order, over up to 2^20 points a slot; a 16-bit table is widened exactly and summed in 32 bits
    return {"rel": 1e-5, "max": 1e-3}
