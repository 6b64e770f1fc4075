"""What a user of the framework has it do, as cases that can be timed.

Most cases are one training step of the compress + error-feedback path: every gradient bucket of a
model through its DDP communication hook, then every Future waited for, as the reducer does.  The
models are those of the benchmark configurations (convolutional nets for CIFAR, a word-level LSTM,
a transformer encoder, a flat 25 MB bucket) and a large fully connected layer; buckets are filled in
reverse order of the parameters up to 25 MiB.  One case is a half-precision count sketch used on its
own, as the compressor classes are by somebody who writes a hook.

A step works in place: it leaves the decompressed gradient in the bucket, and the next pass of the
same state finds it there as its gradient.
"""
import math

import torch

from conef_amd.RandomBlock_hook import RandomBlock_hook, RandomBlockState
from conef_amd.UnbiasedRandomBlock_hook import UnbiasedRandomBlock_hook, UnbiasedRandomBlockState
from conef_amd.compressors.halfCountSketch import DenseCS as HalfDenseCS
from conef_amd.hPowerSGD_hook import hPowerSGDState, hpowerSGD_hook
from conef_amd.powerSGD_hook import PowerSGDState, powerSGD_hook

BUCKET_ELEMENTS = 25 * 1024 * 1024 // 4
BETA = 0.9


# ------------------------------------------------------------------------------ models' parameters
def _resnet(c):
    """CIFAR ResNet: three stages of ``blocks`` pairs of 3x3 convolutions, each with a batch norm."""
    shapes, cin = [(c["width"], 3, 3, 3), (c["width"],), (c["width"],)], c["width"]
    for stage in range(3):
        cout = c["width"] << stage
        for _ in range(2 * c["blocks"]):
            shapes += [(cout, cin, 3, 3), (cout,), (cout,)]
            cin = cout
    return shapes + [(10, cin), (10,)]


def _wide_resnet(c):
    """WRN for CIFAR: ``blocks`` pre-activation blocks a stage, ``width`` times as wide."""
    shapes, cin = [(16, 3, 3, 3)], 16
    for stage in range(3):
        cout = (16 << stage) * c["width"]
        for block in range(c["blocks"]):
            shapes += [(cin,), (cin,), (cout, cin, 3, 3), (cout,), (cout,), (cout, cout, 3, 3)]
            if block == 0:
                shapes.append((cout, cin, 1, 1))
            cin = cout
    return shapes + [(cin,), (cin,), (10, cin), (10,)]


def _lstm(c):
    """Word-level language model: embedding, two LSTM layers, decoder."""
    v, h = c["vocab"], c["hidden"]
    return [(v, h)] + [(4 * h, h), (4 * h, h), (4 * h,), (4 * h,)] * 2 + [(v, h), (v,)]


def _encoder(c):
    """Transformer encoder: embeddings, ``layers`` blocks, pooler and heads."""
    v, h, f = c["vocab"], c["hidden"], c["ffn"]
    shapes = [(v, h), (512, h), (2, h), (h,), (h,)]
    for _ in range(c["layers"]):
        shapes += [(h, h), (h,)] * 4 + [(h,), (h,), (f, h), (f,), (h, f), (h,), (h,), (h,)]
    return shapes + [(h, h), (h,), (h, h), (h,), (h,), (h,), (v,), (2, h), (2,)]


def _matrix(c):
    """One matrix that is a bucket of its own: a flat bucket viewed as rows, a fully connected layer."""
    return [(c["rows"], c["cols"])]


MODELS = {"resnet": _resnet, "wide_resnet": _wide_resnet, "lstm": _lstm, "encoder": _encoder, "matrix": _matrix}


def _numel(shape):
    return math.prod(shape)


def _buckets(shapes):
    out, cur, size = [], [], 0
    for s in reversed(shapes):
        if cur and size + _numel(s) > BUCKET_ELEMENTS:
            out.append(cur)
            cur, size = [], 0
        cur.append(s)
        size += _numel(s)
    return out + [cur] if cur else out


def _matrices(case):
    """(rows, columns) of every gradient the hooks see as a matrix."""
    return [(s[0], _numel(s[1:])) for s in MODELS[case["model"]](case) if len(s) > 1]


class Bucket:
    """What a DDP GradBucket shows a hook: one flat buffer and per-parameter views into it."""

    def __init__(self, flat, shapes, index, is_last):
        self.flat, self.at, self.last, self.views, off = flat, index, is_last, [], 0
        for s in shapes:
            self.views.append(flat[off: off + _numel(s)].view(*s))
            off += _numel(s)

    def buffer(self):
        return self.flat

    def gradients(self):
        return list(self.views)

    def index(self):
        return self.at

    def is_last(self):
        return self.last


# --------------------------------------------------------------------------------------- the cases
def listed():
    bert = dict(model="encoder", vocab=30522, hidden=1024, ffn=4096, layers=4)
    lstm = dict(model="lstm", vocab=33278, hidden=650)
    wrn = dict(model="wide_resnet", blocks=4, width=10)
    return [
        # The smallest step: ResNet-20, 1.1 MB of gradient in one bucket of twenty small matrices.
        dict(name="resnet20 powersgd r2 sketch", path="powersgd", model="resnet", blocks=3, width=16, rank=2, error="sketch",
             sketch_size=0.5),
        # An ordinary one: WRN-28-10, 146 MB in nine buckets, matrices from [160,144] to [640,5760].
        dict(wrn, name="wrn28-10 powersgd r4 sketch", path="powersgd", rank=4, error="sketch", sketch_size=0.2),
        # BERT-large's shapes at four layers (its buckets are alike: more layers are more of the same): low rank on
        # the vector units, high rank on the matrix cores, and the error kept by magnitude instead of sketched.
        dict(bert, name="bert powersgd r8 sketch", path="powersgd", rank=8, error="sketch", sketch_size=0.1),
        dict(bert, name="bert powersgd r32 sketch", path="powersgd", rank=32, error="sketch", sketch_size=0.1),
        dict(bert, name="bert hpowersgd r8 topk", path="hpowersgd", rank=8, error="topk", topk_ratio=0.4),
        # Plain error feedback, the ef_powersgd reducer, on rows of 650 columns (not a multiple of four).
        dict(lstm, name="lstm powersgd r4 dense error", path="powersgd", rank=4, error="dense"),
        # The headline bucket: few rows, far longer than on-chip memory.
        dict(name="flat 25MB randomblock sketch", path="randomblock", model="matrix", rows=5, cols=1_300_000, ratio=0.1,
             error="sketch", sketch_size=0.1),
        # Large embeddings of short rows next to small matrices.
        dict(lstm, name="lstm randomblock sketch", path="randomblock", ratio=0.05, error="sketch", sketch_size=0.1),
        # A fully connected layer (VGG-16 fc6): many rows longer than on-chip memory, the largest bucket there is.
        dict(name="fc6 randomblock sketch", path="randomblock", model="matrix", rows=4096, cols=25088, ratio=0.1,
             error="sketch", sketch_size=0.1),
        # Random blocks with a dense error, the ef_randomblock reducer.
        dict(wrn, name="wrn28-10 randomblock dense error", path="randomblock", ratio=0.1, error="dense"),
        # No error memory at all: the cheapest step per byte of gradient.
        dict(lstm, name="lstm unbiased randomblock", path="unbiased", ratio=0.05),
        # The half-precision sketch as a compressor of its own: unsketch the error onto a gradient, sketch what is left.
        dict(name="half sketch wrn conv", path="half_sketch", model="matrix", rows=640, cols=5760, sketch_size=0.2),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_model(rng, kind):
    if kind == "resnet":
        return dict(model="resnet", blocks=rng.randint(1, 5), width=_log(rng, 8, 24))
    if kind == "wide_resnet":
        return dict(model="wide_resnet", blocks=rng.randint(1, 4), width=_log(rng, 1, 10))
    if kind == "lstm":
        return dict(model="lstm", vocab=_log(rng, 2000, 33278), hidden=_log(rng, 100, 650))
    if kind == "encoder":
        h = _log(rng, 96, 1024)
        return dict(model="encoder", vocab=_log(rng, 2000, 30522), hidden=h, ffn=rng.randint(2 * h, 4 * h),
                    layers=rng.randint(1, 4))
    if kind == "flat":
        rows = rng.randint(1, 8)
        return dict(model="matrix", rows=rows, cols=_log(rng, 50_000, 6_500_000) // rows)
    return dict(model="matrix", rows=_log(rng, 256, 4096), cols=_log(rng, 2000, 25088))


def draw(rng):
    path = rng.choice(["powersgd", "powersgd", "hpowersgd", "randomblock", "randomblock", "unbiased", "half_sketch"])
    if path in ("powersgd", "hpowersgd"):
        case = _draw_model(rng, rng.choice(["resnet", "wide_resnet", "lstm", "encoder"]))
        case.update(path=path, rank=1 << rng.randint(0, 5) if rng.random() < 0.5 else _log(rng, 1, 32))
        if path == "hpowersgd":
            case.update(error="topk", topk_ratio=round(rng.uniform(0.1, 0.6), 3))
        else:
            case.update(error=rng.choice(["sketch", "sketch", "dense"]))
    elif path == "half_sketch":
        case = dict(path=path, model="matrix", rows=_log(rng, 16, 4096), cols=_log(rng, 64, 8192))
    else:
        case = _draw_model(rng, rng.choice(["resnet", "wide_resnet", "lstm", "encoder", "flat", "fc"]))
        case.update(path=path, ratio=round(rng.uniform(0.02, 0.2), 3))
        if path == "randomblock":
            case.update(error=rng.choice(["sketch", "sketch", "dense"]))
    if case.get("error") == "sketch" or path == "half_sketch":
        case["sketch_size"] = round(rng.uniform(0.05, 0.5), 3)
    return case


# ------------------------------------------------------------------------------------ one pass each
def _fill(flat, gen):
    """A gradient as training has it: small entries around zero, one in a hundred from a heavy tail."""
    flat.normal_(0.0, 1e-3, generator=gen)
    u = torch.rand(flat.numel(), generator=gen, device=flat.device)
    tail = u < 0.01
    u = u * 200 - 1                              # on the tail: uniform in [-1, 1)
    flat[tail] = (-1e-2 * torch.sign(u) * torch.log1p(-u.abs().clamp(max=1 - 1e-6)))[tail]


def _hook(case):
    if case["path"] == "powersgd":
        return PowerSGDState(None, matrix_approximation_rank=case["rank"], start_powerSGD_iter=2,
                             use_error_compression=case["error"] == "sketch", sketch_size=case.get("sketch_size", 0.5),
                             beta=BETA), powerSGD_hook
    if case["path"] == "hpowersgd":
        return hPowerSGDState(None, matrix_approximation_rank=case["rank"], start_powerSGD_iter=2, use_error_compression=True,
                              topk_ratio=case["topk_ratio"]), hpowerSGD_hook
    if case["path"] == "randomblock":
        return RandomBlockState(None, compression_ratio=case["ratio"], start_compression_iter=2,
                                use_error_compression=case["error"] == "sketch", sketch_size=case.get("sketch_size", 0.5),
                                beta=BETA), RandomBlock_hook
    return UnbiasedRandomBlockState(None, compression_ratio=case["ratio"], start_compression_iter=2), UnbiasedRandomBlock_hook


class Step:
    """A model in training: its buckets, and the hook's state some iterations in."""

    def __init__(self, case, gen, device):
        self.state, self.hook = _hook(case)
        layout = _buckets(MODELS[case["model"]](case))
        self.buckets = [Bucket(torch.empty(sum(_numel(s) for s in shapes), device=device), shapes, i, i == len(layout) - 1)
                        for i, shapes in enumerate(layout)]
        self.flats = [b.flat for b in self.buckets]
        for _ in range(3):        # two iterations of plain reduction, and the first compressed one, which lays the state out
            for flat in self.flats:
                _fill(flat, gen)
            self.step()
        torch.cuda.synchronize()
        for flat in self.flats:
            _fill(flat, gen)

    def step(self):
        state, hook = self.state, self.hook
        futures = [hook(state, b) for b in self.buckets]
        for f in futures:
            f.wait()

    def __call__(self):
        self.step()
        state = self.state
        out = {"gradient": self.flats}
        for name in ("p_memory_dict", "q_memory_dict", "compressed_tensor_memory"):
            if hasattr(state, name):
                out[name] = getattr(state, name)
        # error memory: one tensor a bucket, or one tensor or sketch a matrix
        errors = []
        for e in getattr(state, "error_dict", {}).values():
            if isinstance(e, torch.Tensor):
                errors.append(e)
            else:
                errors += [getattr(x, "cs", x) for x in (e.values() if isinstance(e, dict) else e)]
        out["error"] = errors
        return out


class HalfSketch:
    """A hook of one's own around the half-precision sketch: the gradient of this iteration, the error
    added to it, and what was not sent (here: everything) put back into the sketch."""

    def __init__(self, case, gen, device):
        self.gradient = torch.empty(case["rows"] * case["cols"], device=device)
        _fill(self.gradient, gen)
        self.gradient = self.gradient.view(case["rows"], case["cols"])
        self.corrected = torch.empty_like(self.gradient)
        self.sketch = HalfDenseCS(case["rows"], case["cols"], case["sketch_size"], device=device)
        self()

    def __call__(self):
        self.corrected.copy_(self.gradient)
        self.sketch.query(self.corrected, 1 - BETA)
        self.sketch.update(self.corrected, BETA)
        return {"corrected": self.corrected, "sketch": self.sketch.cs}


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device).manual_seed(seed)
    return (HalfSketch if case["path"] == "half_sketch" else Step)(case, gen, device)


def run(state):
    return state()


# ------------------------------------------------------------------------------- what a pass is worth
def _width(case, cols):
    return max(int(cols * case["sketch_size"]), 1)


def work(case):
    read_write = flops = 0
    if case["path"] == "half_sketch":
        n, m = case["rows"], case["cols"]
        # gradient read, corrected gradient written, half-precision cells read and written
        return {"bytes": 8 * n * m + 4 * n * _width(case, m), "flops": 5 * n * m}
    for n, m in _matrices(case):
        if case["path"] in ("powersgd", "hpowersgd"):
            r = min(n, m, case["rank"])
            if (n + m) * r * 2 >= n * m:
                # not worth compressing: untouched, except that dense error feedback adds and clears its error
                read_write += 16 * n * m if case["error"] == "dense" else 0
                continue
            read_write += 8 * n * m + 4 * r * (n + 2 * m)       # gradient in and out, P written, Q read and written
            flops += 6 * n * m * r + 2 * n * m
        elif case["path"] == "randomblock":
            read_write += 8 * n * m + 4 * max(1, int(case["ratio"] * n * m))       # gradient in and out, payload written
            flops += n * m
        else:
            k = max(1, int(case["ratio"] * n * m))
            read_write += 4 * n * m + 8 * k        # only the block is read; everything is written, and the payload
            flops += k
            continue
        if case["error"] == "sketch":
            read_write += 8 * n * _width(case, m)
            flops += 4 * n * m
        else:
            read_write += 8 * n * m                # dense error read and written
            flops += 2 * n * m
    return {"bytes": read_write, "flops": flops}


def tolerance(case):
    if case["path"] == "unbiased" or case.get("error") == "dense" and case["path"] == "randomblock":
        return "exact"                             # moves, one addition or one division an element
    if case["path"] == "half_sketch":
        return {"rel": 1e-3, "max": 4e-3}          # cells rounded to eleven bits
    if case["path"] == "hpowersgd":
        # fp32 products and an orthogonalisation; an entry whose magnitude is within rounding of the threshold is
        # kept by one implementation and dropped by another, which is a difference of about the threshold there
        return {"rel": 3e-3, "max": 0.95}
    if case["path"] == "powersgd":
        return {"rel": 3e-5, "max": 2e-3}          # two rounds of fp32 products and orthogonalisations, one fed to the other
    return {"rel": 1e-5, "max": 1e-4}              # sums of fp32 terms in another order
