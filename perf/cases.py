"""Workloads that stand for what a user of trak_amd has it do: featurizing batches of gradients (projection)
and computing attributions from the stored features (X^T X, X (X^T X + lambda I)^-1, scores).

Kinds of cases
  project   CudaProjector.project on one batch of gradients, given as a [rows, features] tensor, as the dict
            of per-parameter tensors a gradient computer returns ("conv": a ResNet-18-style network), or,
            "chunked", as such a dict of a transformer encoder through ChunkedCudaProjector
  xtx       BasicScoreComputer.get_xtx on the features of all training points
  features  BasicScoreComputer.get_x_xtx_inv on them (inverse of the regularized Gram matrix, one product)
  scores    BasicScoreComputer.get_scaled_scores (scores left on the device), or, "to_host", one checkpoint
            through ScoreAccumulator down to the host array of the scores store
  attribute the three steps of a small data set one after another

Sizes: `rows` gradients per batch, `features` gradient length, `proj_dim` JL dimensions, `points` training
points, `targets` target points.
"""
import math

import numpy as np
import torch

from trak_amd import (
    BasicScoreComputer,
    ChunkedCudaProjector,
    CudaProjector,
    ProjectionType,
    ScoreAccumulator,
)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}
DEVICE = "cuda:0"


def conv_shapes(width, classes):
    """Parameter shapes of a ResNet-18 of base width `width` (width 64, 1000 classes: 62 tensors, 11 689 512)."""
    shapes = [(width, 3, 7, 7), (width,), (width,)]
    inp = width
    for out, first in ((width, False), (2 * width, True), (4 * width, True), (8 * width, True)):
        for block in range(2):
            cin = inp if block == 0 else out
            shapes += [(out, cin, 3, 3), (out,), (out,), (out, out, 3, 3), (out,), (out,)]
            if block == 0 and first:
                shapes += [(out, inp, 1, 1), (out,), (out,)]
        inp = out
    return shapes + [(classes, 8 * width), (classes,)]


def encoder_shapes(hidden, layers, vocab):
    """Parameter shapes of a BERT-style encoder with pooler (768, 12, 30 522: 199 tensors, 109 482 240)."""
    shapes = [(vocab, hidden), (512, hidden), (2, hidden), (hidden,), (hidden,)]
    for _ in range(layers):
        shapes += [(hidden, hidden), (hidden,)] * 4 + [(hidden,), (hidden,)]
        shapes += [(4 * hidden, hidden), (4 * hidden,), (hidden, 4 * hidden), (hidden,), (hidden,), (hidden,)]
    return shapes + [(hidden, hidden), (hidden,)]


def chunk_groups(numels, limit):
    """Consecutive parameters grouped into chunks of at most `limit` features: [(begin, end, features)]."""
    groups, begin, width = [], 0, 0
    for i, n in enumerate(numels):
        if width and width + n > limit:
            groups.append((begin, i, width))
            begin, width = i, 0
        width += n
    return groups + [(begin, len(numels), width)]


def parameter_shapes(case):
    if case["layout"] == "conv":
        return conv_shapes(case["width"], case["classes"])
    return encoder_shapes(case["hidden"], case["layers"], case["vocab"])


def gradient_length(case):
    if case["layout"] == "dense":
        return case["features"]
    return sum(math.prod(s) for s in parameter_shapes(case))


def listed():
    return [
        # one query example of a small network (61 706 parameters): scoring single examples as they come in
        {"name": "project_one_example", "kind": "project", "layout": "dense", "rows": 1, "features": 61_706,
         "proj_dim": 512, "dtype": "fp16", "matrix": "rademacher"},
        # full-precision gradients, the configuration that the reference's CPU projector can also run
        {"name": "project_fp32_batch16", "kind": "project", "layout": "dense", "rows": 16, "features": 1_048_576,
         "proj_dim": 512, "dtype": "fp32", "matrix": "rademacher"},
        # batches of eight, the smallest batch option of the projector, of a ResNet-18-sized gradient
        {"name": "project_fp16_batch8", "kind": "project", "layout": "dense", "rows": 8, "features": 11_689_512,
         "proj_dim": 2048, "dtype": "fp16", "matrix": "rademacher"},
        # ResNet-9-sized gradients of CIFAR-style attribution, already flattened
        {"name": "project_fp16_batch32", "kind": "project", "layout": "dense", "rows": 32, "features": 4_825_610,
         "proj_dim": 2048, "dtype": "fp16", "matrix": "rademacher"},
        # ResNet-18 gradients as the gradient computer returns them: a dict of 62 tensors
        {"name": "project_fp16_resnet18_dict", "kind": "project", "layout": "conv", "rows": 32, "width": 64,
         "classes": 1000, "proj_dim": 4096, "dtype": "fp16", "matrix": "rademacher"},
        # BERT-base-sized gradients under a Gaussian matrix, in chunks of parameters: the longest call
        {"name": "project_bf16_bert_normal_chunked", "kind": "project", "layout": "chunked", "rows": 32, "hidden": 768,
         "layers": 12, "vocab": 30_522, "chunk": 27_500_000, "proj_dim": 4096, "dtype": "bf16", "matrix": "normal"},
        # finalize_features of a CIFAR-sized training set in half precision (the default storage type): Gram matrix
        {"name": "xtx_fp16", "kind": "xtx", "points": 50_000, "proj_dim": 2048, "dtype": "fp16"},
        # the same: inverse and product
        {"name": "features_fp16", "kind": "features", "points": 50_000, "proj_dim": 2048, "dtype": "fp16"},
        # full precision at the largest projection dimension in general use
        {"name": "features_fp32", "kind": "features", "points": 50_000, "proj_dim": 4096, "dtype": "fp32"},
        # all test points of such a data set against all training points, full precision: the largest product
        {"name": "scores_fp32", "kind": "scores", "points": 50_000, "targets": 10_000, "proj_dim": 4096,
         "dtype": "fp32", "to_host": False},
        # a handful of test points of interest in half precision, down to the scores store
        {"name": "scores_fp16_few_targets", "kind": "scores", "points": 50_000, "targets": 100, "proj_dim": 2048,
         "dtype": "fp16", "to_host": True},
        # a small study from features to scores
        {"name": "attribute_fp32_small", "kind": "attribute", "points": 2_000, "targets": 100, "proj_dim": 512,
         "dtype": "fp32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, hi):
    return 512 * _log_int(rng, 1, hi // 512)


def draw(rng):
    kind = rng.choice(["dense", "dense", "conv", "chunked", "xtx", "features", "scores", "scores", "attribute"])
    if kind in ("dense", "conv", "chunked"):
        case = {"kind": "project", "layout": kind, "rows": _log_int(rng, 1, 128), "proj_dim": _dim(rng, 4096),
                "dtype": rng.choice(["fp16", "fp16", "bf16", "fp32"]),
                "matrix": rng.choice(["rademacher", "rademacher", "normal"])}
        if kind == "dense":
            case["features"] = _log_int(rng, 10_000, 12_000_000)
        elif kind == "conv":
            case.update(width=8 * rng.randint(1, 8), classes=rng.choice([10, 100, 1000]))
        else:
            case.update(rows=_log_int(rng, 1, 32), hidden=64 * rng.randint(2, 12), layers=rng.randint(2, 12),
                        vocab=30_522, chunk=_log_int(rng, 24_000_000, 80_000_000))
        return case
    dtype = rng.choice(["fp16", "fp32"])
    if kind == "attribute":
        k = _dim(rng, 2048)
        return {"kind": "attribute", "points": _log_int(rng, 2 * k, 10_000), "targets": _log_int(rng, 1, 1_000),
                "proj_dim": k, "dtype": dtype}
    k = _dim(rng, 4096)
    case = {"kind": kind, "points": _log_int(rng, 2 * k, 50_000), "proj_dim": k, "dtype": dtype}
    if kind == "scores":
        case["targets"] = _log_int(rng, 1, 10_000)
        case["to_host"] = case["points"] * case["targets"] <= 20_000_000 and rng.random() < 0.5
    return case


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEVICE)


def _gradients(gen, rows, shapes, dtype, heavy_tails):
    """Per-parameter gradients [rows, ...]: each tensor at its own scale (log-uniform in 1e-5 .. 1e-2), Gaussian, or
    with the tails of a Student t of three degrees of freedom (language models)."""
    scales = (10.0 ** (torch.rand(len(shapes), generator=gen, device=DEVICE) * 3 - 5)).tolist()
    grads = {}
    for i, shape in enumerate(shapes):
        g = _normal(gen, rows, *shape)
        if heavy_tails:
            chi = sum(_normal(gen, rows, *shape).square_() for _ in range(3))
            g *= torch.rsqrt(chi / 3.0)
        grads[f"parameter_{i}"] = (g * scales[i]).to(dtype)
    return grads


def _features(gen, points, proj_dim, dtype):
    return (_normal(gen, points, proj_dim) / math.sqrt(proj_dim)).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    device = torch.device(DEVICE)
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "project":
        rows, k = case["rows"], case["proj_dim"]
        length = gradient_length(case)
        matrix = ProjectionType(case["matrix"])
        if case["layout"] == "dense":
            edges = torch.linspace(0, length, 25).long().tolist()
            grads = torch.empty(rows, length, dtype=dtype, device=device)
            scales = (10.0 ** (torch.rand(24, generator=gen, device=device) * 3 - 5)).tolist()
            for lo, hi, scale in zip(edges, edges[1:], scales):
                grads[:, lo:hi] = _normal(gen, rows, hi - lo) * scale
            projector = CudaProjector(length, k, 7, matrix, device, 32)
        elif case["layout"] == "conv":
            grads = _gradients(gen, rows, parameter_shapes(case), dtype, False)
            projector = CudaProjector(length, k, 7, matrix, device, 32)
        else:
            shapes = parameter_shapes(case)
            grads = _gradients(gen, rows, shapes, dtype, True)
            widths = [g[2] for g in chunk_groups([math.prod(s) for s in shapes], case["chunk"])]
            parts = [CudaProjector(n, k, 123 + i, matrix, device, 32) for i, n in enumerate(widths)]
            projector = ChunkedCudaProjector(parts, case["chunk"], widths, rows, device, dtype)
        return {"kind": "project", "projector": projector, "grads": grads}
    N, k = case["points"], case["proj_dim"]
    state = {"kind": case["kind"], "computer": BasicScoreComputer(dtype=dtype, device=device, lambda_reg=1e-3)}
    x = _features(gen, N, k, dtype)
    if case["kind"] == "scores":
        state.update(features=x, targets=_features(gen, case["targets"], k, dtype), to_host=case["to_host"], dtype=dtype)
        if case["to_host"]:
            state["out_to_loss"] = np.random.default_rng(seed).random((N, 1)).astype(np.float32)
            state["store"] = np.zeros((N, case["targets"]), dtype=np.float16 if dtype == torch.float16 else np.float32)
        else:
            state["out_to_loss"] = torch.rand(N, generator=gen, device=device)
        return state
    state["x"] = x
    if case["kind"] == "features":
        state["xtx"] = (x.float().T @ x.float()).to(dtype)
    if case["kind"] == "attribute":
        state["targets"] = _features(gen, case["targets"], k, dtype)
        state["out_to_loss"] = torch.rand(N, generator=gen, device=device)
    return state


def run(state):
    kind = state["kind"]
    if kind == "project":
        return state["projector"].project(state["grads"], model_id=0)
    computer = state["computer"]
    if kind == "xtx":
        return computer.get_xtx(state["x"])
    if kind == "features":
        return computer.get_x_xtx_inv(state["x"], state["xtx"])
    if kind == "scores":
        features, targets = state["features"], state["targets"]
        if not state["to_host"]:
            return computer.get_scaled_scores(features, targets, state["out_to_loss"])
        accumulator = ScoreAccumulator(computer, features.shape[0], targets.shape[0], dtype=state["dtype"])
        accumulator.add(features, targets, state["out_to_loss"])
        return accumulator.finalize(state["store"])
    xtx = computer.get_xtx(state["x"])
    features = computer.get_x_xtx_inv(state["x"], xtx)
    return {"xtx": xtx, "features": features,
            "scores": computer.get_scaled_scores(features, state["targets"], state["out_to_loss"])}


def work(case):
    """Bytes: every input read once, every output written once.  Operations: 2 rows features proj_dim for a
    projection (making the matrix is not counted), the lower triangle only for the symmetric X^T X, proj_dim^3 for
    the inverse of a symmetric positive definite matrix."""
    e = BYTES[case["dtype"]]
    if case["kind"] == "project":
        length, rows, k = gradient_length(case), case["rows"], case["proj_dim"]
        out = e if case["layout"] == "chunked" else 4
        return {"bytes": rows * length * e + rows * k * out, "flops": 2 * rows * length * k}
    N, k = case["points"], case["proj_dim"]
    xtx = {"bytes": (N * k + k * k) * e, "flops": N * k * (k + 1)}
    features = {"bytes": (2 * N * k + k * k) * e, "flops": 2 * N * k * k + k ** 3}
    if case["kind"] == "xtx":
        return xtx
    if case["kind"] == "features":
        return features
    M = case["targets"]
    out = e if case.get("to_host") else 4
    scores = {"bytes": (N + M) * k * e + N * M * out + 4 * N, "flops": 2 * N * M * k}
    if case["kind"] == "scores":
        return scores
    return {key: xtx[key] + features[key] + scores[key] for key in ("bytes", "flops")}


def tolerance(case):
    """About four times the difference seen between this path and the same path in 64 bits with its results (and
    what it hands from step to step) rounded to the same types."""
    dtype = case["dtype"]
    if case["kind"] == "project":
        if case["layout"] == "chunked":
            # fp32: sums over millions of heavy-tailed values (3e-5 seen); else the result's own rounding
            return {"rel": {"fp16": 5e-4, "bf16": 4e-3, "fp32": 1.2e-4}[dtype]}
        return {"rel": 4e-6}
    if case["kind"] == "xtx":
        return {"rel": {"fp16": 8e-5, "fp32": 1.2e-5}[dtype]}
    if case["kind"] == "features":
        return {"rel": {"fp16": 5e-4, "fp32": 1e-5}[dtype]}
    if case["kind"] == "scores":
        # fp16 scores in the store: a few of them round the other way
        return {"rel": 1e-4 if case["to_host"] and dtype == "fp16" else 4e-6}
    return {"rel": {"fp16": 1.2e-3, "fp32": 2e-5}[dtype]}
