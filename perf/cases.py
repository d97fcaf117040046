"""The work whose speed is measured: what programs built with this package spend their calls on.

Every case is one of the package's benchmark programs (``functs_amd.benchmark.PROGRAMS``) called the
way a user calls it - scripted, built once for its shapes, called again and again on new tensors - or
the detection tail as an operator of its own.  Each program is listed at one size of its range; the
detection filter, the elementwise loop and the recurrence, which are used over wide ranges, at two
or three."""
import math
from statistics import NormalDist

import torch

import functs_amd.jit as fj
from functs_amd.benchmark import PROGRAMS
from functs_amd.benchmark.inputs import YOLO_BASE_SIZES, yolo_anchors

CONF_LOGIT = math.log(0.3 / 0.7)      # the detection filter keeps sigmoid(objectness) >= 0.3


def listed():
    return [
        # the get_started example, an in-place loop over the rows of a matrix, at an odd size: the
        # cheapest call, bound by its launch and by the host
        {"name": "loop_3001x1111", "program": "c1", "rows": 3001, "cols": 1111, "dtype": "float32"},
        # the same loop over an activation-sized matrix in the type that activations have: bandwidth
        {"name": "loop_8192_bf16", "program": "c1", "rows": 8192, "cols": 4096, "dtype": "bfloat16"},
        # detection filter, one 416 x 416 image, 80 classes: online inference
        {"name": "yolo_1x416", "program": "c2", "batch": 1, "size": 416, "classes": 80, "trained": False},
        # the same over a batch in a per-image loop: the benchmark's headline workload
        {"name": "yolo_16x416", "program": "c5", "batch": 16, "size": 416, "classes": 80, "trained": False},
        # larger images, a data set of one's own, and a trained head: few rows pass the filter
        {"name": "yolo_12x608_c13", "program": "c5", "batch": 12, "size": 608, "classes": 13, "trained": True},
        # SSD300 post-processing: decode, softmax, per-class filter; the classes are joined for what follows
        {"name": "ssd_8732", "program": "c3", "priors": 8732, "classes": 81},
        # stacked LSTM, one sequence: a chain of dependent steps
        {"name": "lstm_1x512", "program": "c4", "steps": 64, "batch": 1, "hidden": 512, "layers": 2},
        # a batch of sequences through a smaller stack
        {"name": "lstm_8x256", "program": "c4", "steps": 100, "batch": 8, "hidden": 256, "layers": 3},
        # a whole detection head as a model's forward has it, from NCHW maps to the boxes behind the NMS
        {"name": "head_nms_4x608", "program": "yolo_head_nms", "batch": 4, "size": 608, "classes": 80},
        # proposals of one image through class-aware NMS
        {"name": "nms_2000", "program": "batched_nms", "boxes": 2000, "objects": 60, "clutter": 200, "classes": 20},
        # decoding with a growing key / value cache
        {"name": "attention_12x50", "program": "attention", "batch": 1, "heads": 12, "length": 50, "start": 32},
        # class-wise box regression of every prior
        {"name": "delta2bbox_8732x21", "program": "delta2bbox", "boxes": 8732, "classes": 21},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    program = rng.choice(["c1", "c1", "c2", "c5", "c5", "c3", "c4", "c4", "yolo_head_nms", "batched_nms", "attention", "delta2bbox"])
    if program == "c1":
        return {"program": "c1", "rows": _log(rng, 16, 8192), "cols": _log(rng, 16, 4096), "dtype": rng.choice(["float32", "float32", "float16", "bfloat16"])}
    if program == "c2":
        return {"program": "c2", "batch": 1, "size": 32 * rng.randint(7, 20), "classes": _log(rng, 1, 91), "trained": rng.random() < 0.5}
    if program == "c5":
        # (three results an image)
        batch, classes = rng.randint(2, 20), _log(rng, 1, 91)
        most = 16 * 10647 * 85 / (batch * (5 + classes))     # rows of an image, so that a call reads no more than the headline workload
        size = max(s for s in range(224, 641, 32) if s == 224 or 63 * (s // 32) ** 2 <= most)
        return {"program": "c5", "batch": batch, "size": 32 * rng.randint(7, size // 32), "classes": classes, "trained": rng.random() < 0.5}
    if program == "c3":
        return {"program": "c3", "priors": _log(rng, 500, 24564), "classes": rng.randint(2, 91)}
    if program == "c4":
        hidden = 2 ** rng.randint(6, 9)
        return {"program": "c4", "steps": _log(rng, 8, 100), "batch": _log(rng, 1, 8), "hidden": hidden, "layers": rng.randint(1, 3)}
    if program == "yolo_head_nms":
        return {"program": "yolo_head_nms", "batch": rng.randint(1, 4), "size": 32 * rng.randint(7, 19), "classes": _log(rng, 10, 80)}
    if program == "batched_nms":
        boxes = _log(rng, 100, 2000)
        return {"program": "batched_nms", "boxes": boxes, "objects": _log(rng, 5, 60), "clutter": rng.randint(0, boxes // 8), "classes": _log(rng, 1, 80)}
    if program == "attention":
        steps = rng.randint(4, 18)
        length = rng.randint(steps + 8, 96)
        return {"program": "attention", "batch": rng.randint(1, 4), "heads": rng.choice([4, 6, 8, 12]), "length": length, "start": length - steps}
    return {"program": "delta2bbox", "boxes": _log(rng, 50, 8732), "classes": _log(rng, 1, 21)}


_built = {}


def _build(case, args):
    """A program is scripted and built once for its shapes and kept, as the program around it keeps it."""
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    fn = _built.get(key)
    if fn is None:
        fn = _built[key] = fj.build(fj.script(PROGRAMS[case["program"]]), args)
    return fn


def _anchors(size):
    cells = size // 32
    anchors, strides = yolo_anchors((cells, 2 * cells, 4 * cells))
    return anchors.cuda(), strides.cuda()


def _rows(size):
    return 63 * (size // 32) ** 2     # three anchors on grids of s, 2 s and 4 s cells a side


def _above(x):
    """Share of N(0, 1) above x."""
    return 0.5 * math.erfc(x / math.sqrt(2.0))


def _kept(case):
    """Rows of every image that pass the detection filter: as many as of N(0, 1) logits, or with a
    trained head about two in a hundred, in some images more than in others."""
    rows, batch = _rows(case["size"]), case["batch"]
    if not case["trained"]:
        return [round(rows * _above(CONF_LOGIT))] * batch
    return [max(1, round(rows * 0.02 * (0.5 + (i + 0.5) / batch))) for i in range(batch)]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    program = case["program"]
    if program == "c1":
        dtype = getattr(torch, case["dtype"])
        b = normal(case["rows"], case["cols"]).to(dtype)
        args = [b[:1].clone(), b, case["rows"]]
    elif program in ("c2", "c5"):
        anchors, strides = _anchors(case["size"])
        pred = normal(case["batch"], anchors.size(0), 5 + case["classes"])
        objectness = pred[..., 4]
        if case["trained"]:
            objectness.mul_(1.5)
        # every image's logits are moved so that the number of its rows above the threshold does not
        # depend on the seed, and kept clear of the threshold itself
        order = objectness.sort(dim=1, descending=True).values
        for image, kept in enumerate(_kept(case)):
            objectness[image] += CONF_LOGIT - 0.5 * (order[image, kept - 1] + order[image, kept])
        objectness += 1e-3 * (objectness - CONF_LOGIT).sign()
        args = [pred, anchors, strides]
    elif program == "c3":
        # the same rows of class logits in another order: how many pass the filter does not depend on the seed
        fixed = torch.Generator(device="cuda").manual_seed(0)
        conf = torch.randn(case["priors"], case["classes"], generator=fixed, device="cuda")
        conf = conf[torch.randperm(case["priors"], generator=g, device="cuda")]
        args = [0.5 * normal(1, case["priors"], 4), conf[None], uniform(case["priors"], 4)]
    elif program == "c4":
        steps, batch, hidden, layers = case["steps"], case["batch"], case["hidden"], case["layers"]
        weights = [uniform(*s) * 0.2 - 0.1 for s in ((layers, 4, hidden, hidden), (layers, 4, hidden, hidden), (layers, 4, 1, hidden), (layers, 4, 1, hidden))]
        args = [normal(steps, batch, hidden)] + weights
    elif program == "yolo_head_nms":
        cells, attributes = case["size"] // 32, 5 + case["classes"]
        maps = [normal(case["batch"], 3 * attributes, f, f) for f in (cells, 2 * cells, 4 * cells)]
        for m in maps:
            # class logits as behind a trained head: about 700 scores an image pass the tail's threshold of 0.05
            shift = math.log(0.05 / 0.95) + NormalDist().inv_cdf(700.0 / (_rows(case["size"]) * case["classes"]))
            m.view(case["batch"], 3, attributes, m.size(2), m.size(3))[:, :, 5:] += shift
        bases = []
        for level, stride in enumerate((32, 16, 8)):
            half = torch.tensor(YOLO_BASE_SIZES[level], dtype=torch.float32) * 0.5
            bases.append(torch.cat([stride / 2.0 - half, stride / 2.0 + half], dim=1).cuda())
        args = [maps, bases]
    elif program == "batched_nms":
        # proposals as a detector emits them: every object is hit by many boxes that overlap, clutter by
        # one; each in a cell of its own, so that the number of survivors does not depend on the seed
        n, objects, clutter = case["boxes"], case["objects"], case["clutter"]
        cells = math.isqrt(objects + clutter - 1) + 1
        cell = torch.randperm(cells * cells, generator=g, device="cuda")[:objects + clutter]
        which = torch.arange(n, device="cuda")
        which = torch.where(which < clutter, objects + which, which % objects)[torch.randperm(n, generator=g, device="cuda")]
        middle = torch.stack([cell % cells, cell // cells], dim=1)[which] * 128.0 + 64.0
        half = (uniform(objects + clutter, 2) * 36 + 12)[which]
        centre = middle + half * 0.1 * (uniform(n, 2) - 0.5)
        half = half * (1 + 0.2 * (uniform(n, 2) - 0.5))
        boxes = torch.cat([centre - half, centre + half], dim=1)
        labels = torch.randint(0, case["classes"], (objects + clutter,), generator=g, device="cuda")[which]
        return {"fn": torch.ops.functs.batched_nms, "args": [boxes, uniform(n), labels, 0.45]}
    elif program == "attention":
        batch, heads, length, start, depth = case["batch"], case["heads"], case["length"], case["start"], 64
        k, v = torch.zeros(batch, heads, length, depth, device="cuda"), torch.zeros(batch, heads, length, depth, device="cuda")
        k[:, :, :start], v[:, :, :start] = normal(batch, heads, start, depth), normal(batch, heads, start, depth)
        bound = (6.0 / (2 * depth)) ** 0.5
        args = [normal(batch, heads, 1, depth), k, v] + [(uniform(heads, depth, depth) * 2 - 1) * bound for _ in range(4)] + [start]
    else:
        rois = uniform(case["boxes"], 4) * 150
        rois[:, 2:] += rois[:, :2]
        args = [rois, normal(case["boxes"], 4 * case["classes"])]
    return {"fn": _build(case, args), "args": args, "join": program == "c3"}


def run(state):
    out = state["fn"](*state["args"])
    if state.get("join"):
        # the classes' boxes and scores as one tensor each, which is what the tail behind them takes
        return torch.cat(out[0]), torch.cat(out[1])
    return out


def work(case):
    program = case["program"]
    if program == "c1":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * (4 if case["dtype"] == "float32" else 2), "flops": n}
    if program in ("c2", "c5"):
        # the objectness of every row; the rest of the row, its anchor and its stride only for rows that are kept
        rows, width = case["batch"] * _rows(case["size"]), 5 + case["classes"]
        kept = sum(_kept(case))
        tables = min(kept, _rows(case["size"])) * 20
        return {"bytes": 4 * rows + 4 * (width - 1) * kept + tables + 4 * width * kept, "flops": 4 * rows + (4 * width + 20) * kept}
    if program == "c3":
        n, classes = case["priors"], case["classes"]
        kept = n * (classes - 1) * _above(math.log(0.05 * classes) + 0.5)
        return {"bytes": 4 * n * (8 + classes) + 2 * 20 * kept, "flops": n * (5 * classes + 20)}
    if program == "c4":
        steps, batch, hidden, layers = case["steps"], case["batch"], case["hidden"], case["layers"]
        weights = layers * 8 * hidden * (hidden + 1)
        return {"bytes": 4 * (weights + 2 * steps * batch * hidden + 2 * layers * batch * hidden), "flops": 16 * steps * batch * layers * hidden * hidden}
    if program == "yolo_head_nms":
        rows, width = case["batch"] * _rows(case["size"]), 5 + case["classes"]
        return {"bytes": 4 * rows * width + case["batch"] * 100 * 28, "flops": rows * (4 * width + 20)}
    if program == "batched_nms":
        n, kept = case["boxes"], case["objects"] + case["clutter"]
        return {"bytes": n * 28 + kept * 28, "flops": 6 * n * kept + n * math.log2(n)}
    if program == "attention":
        lanes, length, depth = case["batch"] * case["heads"], case["length"], 64
        return {"bytes": 4 * (lanes * (4 * length * depth + 2 * depth) + 4 * case["heads"] * depth * depth),
                "flops": (length - case["start"]) * lanes * (8 * depth * depth + 4 * length * depth)}
    n = case["boxes"] * case["classes"]
    return {"bytes": 4 * (4 * case["boxes"] + 8 * n), "flops": 30 * n}


def tolerance(case):
    # Four times what the programs differ by from themselves in 64 bits: 4e-8 to 1.2e-7 (largest 3.7e-7)
    # where values are only decoded, 1.9e-7 (largest 1.6e-6) through sums and dependent steps.
    # Additions of 1 and selected boxes are the same bits.
    program = case["program"]
    if program in ("c1", "batched_nms"):
        return "exact"
    if program in ("c4", "attention"):
        return {"rel": 8e-7, "max": 8e-6}
    return {"rel": 5e-7, "max": 2e-6}
