"""What the performance of this framework is measured on: training steps, validation passes and weight
updates of pipeline stages, each driven the way a training program drives them.

A case is a dict of plain values; ``kind`` selects one of the programs below, the other entries are its sizes.
``prepare`` builds what such a program holds before the step (stages, optimizers with their version rings, data on
the GPU, the forward passes of a filled pipeline), ``run`` is one step of it.  Activations that a backward pass
needs later are counted in ``work`` as written once and read once: no cache holds them until then.
"""
import contextlib
import math

import torch

from pipedream_amd import adam, handoff, layers, optimizer, runtime, schedule, sgd
from pipedream_amd.stages import gnmt, mlp, transformer, vgg16

SGD_ARGS = dict(lr=0.01, momentum=0.9, weight_decay=5e-4)
# (all of VGG16 from random weights on random labels: at 0.01 two correct fp32 implementations are 10 % apart after
# three steps, at a fine-tuning rate they stay as close as they are after the first)
VGG16_SGD_ARGS = dict(SGD_ARGS, lr=1e-4)
ADAM_ARGS = dict(lr=1e-3, betas=(0.9, 0.999))
PAD = 0                                       # padding token of the translation stages

# (in, out channels, side of the image at 224 x 224) of VGG16's convolutions; Linear layers below
VGG_CONVS = [(3, 64, 224), (64, 64, 224), (64, 128, 112), (128, 128, 112), (128, 256, 56), (256, 256, 56),
             (256, 256, 56), (256, 512, 28), (512, 512, 28), (512, 512, 28), (512, 512, 14), (512, 512, 14),
             (512, 512, 14)]
VGG_LINEARS = [(25088, 4096), (4096, 4096), (4096, 1000)]
VGG_PARAMS = 138357544


def listed():
    return [
        # the small end: a two-stage MLP pipeline, where launches and host time are everything
        dict(name="mlp_b32", kind="mlp", batch=32, d_in=784, d_hidden=1024, d_out=10),
        # conv1_1 .. pool2 of VGG16 as one stage of a pipeline of depth 4: the headline workload
        dict(name="vgg_front_b64", kind="vgg_front", batch=64, height=224, width=224),
        # the same stage on a small batch of odd-sized images (fine-tuning on crops)
        dict(name="vgg_front_odd", kind="vgg_front", batch=7, height=101, width=147),
        # all of VGG16 as four stages that share the GPU, stash depths 4/3/2/1: the largest
        dict(name="vgg16_b64", kind="vgg16", batch=64, plain_handoff=False),
        # validation of the same pipeline on a few images: forward passes only
        dict(name="vgg16_eval_b8", kind="vgg16_eval", batch=8, minibatches=2),
        # embedding + 4 LSTM layers at the size of the GNMT configuration, forward beside backward
        dict(name="gnmt_t50_b128", kind="gnmt", steps=50, batch=128, hidden=1024, vocab=32320, overlap=True),
        # the stage with the bidirectional first layer on ragged sentences, one stream
        dict(name="gnmt_bidir_t31_b40", kind="gnmt_bidir", steps=31, batch=40, hidden=1024, vocab=32320),
        # classifier + label smoothing, the tail of the last translation stage
        dict(name="gnmt_head_t50_b128", kind="gnmt_head", steps=50, batch=128, hidden=1024, vocab=32320),
        # six transformer layers, bf16 with fp32 masters, four micro-batches and one Adam update
        dict(name="transformer_b8_s512", kind="transformer", batch=8, seq=512, hidden=1024, depth=6, overlap=True),
        # sequences that are no power of two and few of them, a narrower model
        dict(name="transformer_b3_s200", kind="transformer", batch=3, seq=200, hidden=768, depth=4, overlap=False),
        # a validation pass over one short sequence: launch-bound
        dict(name="transformer_eval_b1_s128", kind="transformer_eval", batch=1, seq=128, hidden=1024, depth=6),
        # the stashed Adam update of a large stage by itself: memory-bound
        dict(name="adam_vgg16_params", kind="update", rule="adam", mixed=False, params=VGG_PARAMS, tensors=32),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["mlp", "vgg_front", "vgg16", "vgg16_eval", "gnmt", "gnmt_bidir", "gnmt_head", "transformer",
                       "transformer", "transformer_eval", "update"])
    if kind == "mlp":
        return dict(kind=kind, batch=_log_uniform(rng, 16, 512), d_in=_log_uniform(rng, 64, 2048),
                    d_hidden=_log_uniform(rng, 128, 2048), d_out=_log_uniform(rng, 10, 1000))
    if kind == "vgg_front":
        height, width = rng.randint(32, 224), rng.randint(32, 224)
        return dict(kind=kind, batch=_log_uniform(rng, 1, 64), height=height, width=width)
    if kind == "vgg16":                        # (with fewer images a single ReLU decision is a large share of a gradient)
        return dict(kind=kind, batch=_log_uniform(rng, 16, 60), plain_handoff=rng.random() < 0.5)
    if kind == "vgg16_eval":
        return dict(kind=kind, batch=_log_uniform(rng, 1, 60), minibatches=rng.randint(1, 4))
    if kind in ("gnmt", "gnmt_bidir"):
        case = dict(kind=kind, steps=rng.randint(5, 50), batch=_log_uniform(rng, 8, 128),
                    hidden=rng.choice([512, 768, 1024]), vocab=rng.randint(8000, 32320))
        if kind == "gnmt":
            case["overlap"] = rng.random() < 0.5
        return case
    if kind == "gnmt_head":
        return dict(kind=kind, steps=rng.randint(5, 50), batch=_log_uniform(rng, 8, 128),
                    hidden=rng.choice([512, 768, 1024]), vocab=8 * rng.randint(1000, 4040))
    if kind in ("transformer", "transformer_eval"):
        case = dict(kind=kind, batch=_log_uniform(rng, 1, 8), seq=8 * _log_uniform(rng, 4, 80),
                    hidden=rng.choice([512, 768, 1024]), depth=rng.randint(1, 6))
        if kind == "transformer":
            case["overlap"] = rng.random() < 0.5
        return case
    return dict(kind=kind, rule=rng.choice(["adam", "sgd"]), mixed=rng.random() < 0.5,
                params=_log_uniform(rng, 200000, VGG_PARAMS), tensors=rng.randint(4, 40))


# -- the programs -----------------------------------------------------------------------------------------------

class _Pipeline(object):
    """Stages that share the GPU in steady-state 1F1B: one step takes every stage through one forward pass, one
    backward pass and one stashed SGD update, last stage first, so that each stage finds its neighbour's gradient
    and its producer's activation queued."""

    def __init__(self, model, conf, batches, sgd_args=None):
        handoff.reset_fabrics()                    # a pipeline of its own beside any that is still alive
        ranks = len(conf["stage_to_rank_map"])
        x, target = batches[0]
        shapes = {"input0": tuple(x.shape), "target": tuple(target.shape)}
        dtypes = {"input0": torch.float32, "target": torch.int64}
        maps = dict(conf, stage_to_depth_map=None)
        self.batches = batches
        self.stages = [runtime.StageRuntime(
            model=model, distributed_backend="gloo", fp16=False, loss_scale=1.0, training_tensor_shapes=shapes,
            eval_tensor_shapes=dict(shapes), training_tensor_dtypes=dtypes, inputs_module_destinations={"input": 0},
            target_tensor_names={"target"}, configuration_maps=maps, master_addr="127.0.0.1", rank=rank, local_rank=0,
            num_ranks_in_server=ranks, verbose_freq=0, model_type=runtime.IMAGE_CLASSIFICATION)
            for rank in range(ranks)]
        if sgd_args is None:                       # validation
            return
        self.optimizers = [sgd.SGDWithWeightStashing(r.modules(), r.master_parameters, r.model_parameters, 1.0,
                                                     num_versions=r.num_warmup_minibatches + 1, **sgd_args)
                           for r in self.stages]
        for r in self.stages:
            r.train(1 << 30)
            r.set_loader(self.endless() if r.stage == 0 else None)
        for r in self.stages:                      # fill: W forward passes in flight in every stage
            for _ in range(r.num_warmup_minibatches):
                r.run_forward()

    def endless(self):
        while True:
            for batch in self.batches:
                yield batch

    def run(self):
        for r, opt in zip(reversed(self.stages), reversed(self.optimizers)):
            r.run_forward()
            opt.zero_grad()
            opt.load_old_params()
            r.run_backward()
            opt.load_new_params()
            opt.step()
        last = self.stages[-1]
        return {"loss": last.loss, "logits": last.output,
                "grads": [p.grad for r in self.stages for p in r.parameters()]}


class _Evaluation(_Pipeline):
    """Validation of the pipeline: forward passes under the acknowledgement clock, no optimizer."""

    def run(self):
        seen = []
        last = self.stages[-1]
        with torch.no_grad():
            schedule.run_pipeline([schedule.stage_eval_loop(
                r, len(self.batches), self.batches,
                on_forward=(lambda i, r: seen.append((r.output, r.loss))) if r is last else None)
                for r in self.stages])
        return seen


class _Neighbours(torch.nn.Module):
    """Stands for the stages behind the one that is run."""

    def forward(self, x):
        raise RuntimeError("the stages behind this one are played by the caller")


class _FrontStage(object):
    """The first stage of a pipeline of depth 4, with its neighbour played through the hand-off queues."""

    def __init__(self, case, generator):
        handoff.reset_fabrics()
        with torch.device("cuda"):
            model = [(vgg16.FrontStage(), ["input0"], ["out0"]), (_Neighbours(), ["out0"], ["out1"]),
                     (layers.CrossEntropyLoss(), ["out1"], ["loss"])]
        b, h, w = case["batch"], case["height"], case["width"]
        out = (b, 128, h // 4, w // 4)
        shapes = {"input0": (b, 3, h, w), "target": (b,), "out0": out}
        dtypes = {"input0": torch.float32, "target": torch.int64, "out0": torch.float32}
        self.r = runtime.StageRuntime(
            model=model, distributed_backend="gloo", fp16=False, loss_scale=1.0, training_tensor_shapes=shapes,
            eval_tensor_shapes=dict(shapes), training_tensor_dtypes=dtypes, inputs_module_destinations={"input": 0},
            target_tensor_names={"target"},
            configuration_maps={"module_to_stage_map": [0, 1, 1], "stage_to_rank_map": {"0": [0], "1": [1]},
                                "stage_to_depth_map": {"0": 3, "1": 0}},
            master_addr="127.0.0.1", rank=0, local_rank=0, num_ranks_in_server=2, verbose_freq=0,
            model_type=runtime.IMAGE_CLASSIFICATION)
        self.opt = sgd.SGDWithWeightStashing(self.r.modules(), self.r.master_parameters, self.r.model_parameters, 1.0,
                                             num_versions=4, **SGD_ARGS)
        self.batches = [(_images(b, h, w, generator), _classes(b, 1000, generator)) for _ in range(2)]
        self.upstream = _normal(out, generator, 1e-3).contiguous(memory_format=torch.channels_last)
        self.r.train(1 << 30)
        self.r.set_loader(_Pipeline.endless(self))
        for _ in range(3):
            self.forward()

    def forward(self):
        self.r.run_forward()
        fabric = self.r.comm_handler.fabric
        out = fabric.take("out0", 1, False).tensor
        fabric.take("target", 1, False)
        fabric.put("out0", 0, True, self.upstream)
        return out

    def run(self):
        out = self.forward()
        self.opt.zero_grad()
        self.opt.load_old_params()
        self.r.run_backward()
        self.opt.load_new_params()
        self.opt.step()
        return {"out": out, "grads": [p.grad for p in self.r.parameters()], "updated": list(self.r.parameters())}


class _Streams(object):
    """One stream for everything, or (``overlap``) one per minibatch in flight."""

    def __init__(self, warmup, overlap):
        self.ring = schedule.MinibatchStreams(warmup) if overlap else None
        if overlap:
            self.ring.join()

    def forward(self, minibatch):
        return self.ring.forward(minibatch) if self.ring is not None else contextlib.nullcontext()

    def backward(self, minibatch):
        return self.ring.backward(minibatch) if self.ring is not None else contextlib.nullcontext()

    def leave(self):
        if self.ring is not None:
            self.ring.leave()


class _Translation(object):
    """A translation stage with two forward passes in flight: Adam with three weight versions."""

    def __init__(self, case, generator):
        steps, batch, hidden = case["steps"], case["batch"], case["hidden"]
        bidirectional = case["kind"] == "gnmt_bidir"
        with torch.device("cuda"):
            self.module = (gnmt.BidirStage0 if bidirectional else gnmt.Stage0)(case["vocab"], hidden)
        self.params = list(self.module.parameters())
        self.opt = adam.AdamWithWeightStashing([self.module], self.params, None, 1.0, 3, **ADAM_ARGS)
        ids, lengths = _sentences(steps, batch, case["vocab"], generator, ragged=bidirectional)
        self.inputs = (ids, lengths) if bidirectional else (ids,)
        self.upstream = [_normal((steps, batch, hidden), generator, 1e-2) for _ in range(2 if bidirectional else 1)]
        self.streams = _Streams(2, case.get("overlap", False))
        self.started = self.finished = 0
        self.pending = []
        for _ in range(2):
            self.forward()

    def forward(self):
        with self.streams.forward(self.started):
            out = self.module(*self.inputs)
        self.pending.append(out if isinstance(out, tuple) else (out,))
        self.started += 1

    def run(self):
        self.forward()
        out = self.pending.pop(0)
        with self.streams.backward(self.finished):
            self.opt.zero_grad()
            self.opt.load_old_params()
            torch.autograd.backward(out, self.upstream)
            self.opt.load_new_params()
            self.opt.step()
        self.finished += 1
        self.streams.leave()
        return {"out": [t.detach() for t in out], "grads": [p.grad for p in self.params]}


class _TranslationHead(object):
    """Classifier and criterion of the last translation stage, which keeps one weight version."""

    def __init__(self, case, generator):
        steps, batch, hidden, vocab = case["steps"], case["batch"], case["hidden"], case["vocab"]
        with torch.device("cuda"):
            self.module = layers.Linear(hidden, vocab)
        self.criterion = layers.LabelSmoothing(PAD, 0.1)
        self.opt = adam.AdamWithWeightStashing([self.module], list(self.module.parameters()), None, 1.0, 1, **ADAM_ARGS)
        self.x = torch.tanh(_normal((steps, batch, hidden), generator)).requires_grad_()
        self.target = _sentences(steps, batch, vocab, generator, ragged=True)[0].view(-1)

    def run(self):
        logits = self.module(self.x)
        loss = self.criterion(logits, self.target)
        self.opt.zero_grad()
        self.opt.load_old_params()
        self.x.grad = None
        loss.backward()
        self.opt.load_new_params()
        self.opt.step()
        return {"loss": loss.detach(), "dx": self.x.grad, "grads": [p.grad for p in self.module.parameters()]}


class _Transformer(object):
    """A transformer stage with double-buffered weights: four micro-batches and one update a step."""

    MICRO_BATCHES = 4

    def __init__(self, case, generator):
        batch, seq, hidden = case["batch"], case["seq"], case["hidden"]
        with torch.device("cuda"):
            self.module = transformer.Stage0(case["depth"], hidden, hidden // 64, 4 * hidden)
        self.opt = adam.AdamWithWeightStashing([self.module], list(self.module.parameters()), None, 1.0, 2,
                                               update_interval=self.MICRO_BATCHES, bf16_image=True, **ADAM_ARGS)
        self.x = [_normal((batch, seq, hidden), generator) for _ in range(self.MICRO_BATCHES)]
        self.upstream = _normal((batch, seq, hidden), generator, 0.05).bfloat16()
        if case["kind"] == "transformer_eval":
            return
        self.streams = _Streams(1, case["overlap"])
        self.started = self.finished = 0
        self.pending = []
        self.forward()

    def forward(self):
        x = self.x[self.started % self.MICRO_BATCHES].detach().requires_grad_()      # as the hand-off gives it
        with self.streams.forward(self.started):
            self.pending.append((x, self.module(x)))
        self.started += 1

    def run(self):
        for _ in range(self.MICRO_BATCHES):
            self.forward()
            x, out = self.pending.pop(0)
            with self.streams.backward(self.finished):
                self.opt.zero_grad()
                self.opt.load_old_params()
                out.backward(self.upstream)
                self.opt.load_new_params()
                self.opt.step()
            self.finished += 1
        self.streams.leave()
        # (the gradients of the LayerNorm shifts are left out: six layers have more than 64 of everything)
        return {"out": out.detach(), "dx": x.grad,
                "grads": [p.grad for n, p in self.module.named_parameters() if not n.endswith(("ln1.bias", "ln2.bias"))]}


class _TransformerEval(_Transformer):
    def run(self):
        with torch.no_grad():
            return self.module(self.x[0])


class _Update(object):
    """The stashed update by itself, two weight versions; ``mixed``: bf16 model parameters with fp32 masters."""

    def __init__(self, case, generator):
        # a stage's parameters: matrices and the vectors that go with them, sizes falling off like 1 / rank
        count = case["tensors"]
        weights = [1.0 / (1 + i // 2) if i % 2 == 0 else 0.002 for i in range(count)]
        sizes = [max(1, int(case["params"] * w / sum(weights))) for w in weights]
        with torch.device("cuda"):
            self.module = torch.nn.ParameterList([torch.nn.Parameter(_normal((n,), generator, 0.02)) for n in sizes])
        masters, model = list(self.module), None
        if case["mixed"]:
            self.module = self.module.bfloat16()
            model, masters = optimizer.prep_param_lists(self.module)
        build, args = ((adam.AdamWithWeightStashing, ADAM_ARGS) if case["rule"] == "adam"
                       else (sgd.SGDWithWeightStashing, SGD_ARGS))
        self.opt = build([self.module], masters, model, 128.0 if case["mixed"] else 1.0, 2, **args)
        self.masters = masters
        for p in self.module:
            p.grad = _normal(p.shape, generator, 1e-3).to(p.dtype)

    def run(self):
        self.opt.load_new_params()
        self.opt.step()
        return list(self.masters)


# -- data -------------------------------------------------------------------------------------------------------

def _normal(shape, generator, scale=1.0):
    return torch.randn(shape, generator=generator, device="cuda") * scale


def _images(batch, height, width, generator):
    return _normal((batch, 3, height, width), generator).contiguous(memory_format=torch.channels_last)


def _classes(batch, classes, generator):
    return torch.randint(0, classes, (batch,), generator=generator, device="cuda")


def _sentences(steps, batch, vocab, generator, ragged):
    """Token ids [steps, batch], padded behind each sentence's end, and the lengths (longest first)."""
    ids = torch.randint(1, vocab, (steps, batch), generator=generator, device="cuda")
    low = max(1, steps // 2) if ragged else steps
    lengths = torch.randint(low, steps + 1, (batch,), generator=generator, device="cuda").sort(descending=True)[0]
    lengths[0] = steps
    ids[torch.arange(steps, device="cuda")[:, None] >= lengths[None, :]] = PAD
    return ids, lengths


def prepare(case, seed):
    torch.manual_seed(seed)                        # initial weights, and the dropout masks drawn during the step
    generator = torch.Generator("cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "mlp":
        with torch.device("cuda"):
            model = mlp.model(layers.CrossEntropyLoss(), case["d_in"], case["d_hidden"], case["d_out"])
        batches = [(torch.rand(case["batch"], case["d_in"], generator=generator, device="cuda"),
                    _classes(case["batch"], case["d_out"], generator)) for _ in range(2)]
        return _Pipeline(model, mlp.conf(), batches, SGD_ARGS)
    if kind in ("vgg16", "vgg16_eval"):
        with torch.device("cuda"):
            model = vgg16.model(layers.CrossEntropyLoss(), plain_handoff=case.get("plain_handoff", False))
        batches = [(_images(case["batch"], 224, 224, generator), _classes(case["batch"], 1000, generator))
                   for _ in range(case.get("minibatches", 2))]
        if kind == "vgg16_eval":
            return _Evaluation(model, vgg16.conf(), batches)
        return _Pipeline(model, vgg16.conf(), batches, VGG16_SGD_ARGS)
    return {"vgg_front": _FrontStage, "gnmt": _Translation, "gnmt_bidir": _Translation, "gnmt_head": _TranslationHead,
            "transformer": _Transformer, "transformer_eval": _TransformerEval, "update": _Update}[kind](case, generator)


def run(state):
    return state.run()


# -- what a pass cannot do without ------------------------------------------------------------------------------

def _training(params, stored, flops, bytes_per_param, io=0.0):
    """Bytes and flops of a training step: activations written and read once, weights read by the forward and the
    backward pass, gradients written, and the update."""
    return {"bytes": 8.0 * stored + params * (8 + 4 + bytes_per_param) + io, "flops": float(flops)}


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        b, i, h, o = case["batch"], case["d_in"], case["d_hidden"], case["d_out"]
        params = i * h + h * h + h * o + 2 * h + o
        return _training(params, b * (i + 2 * h + o), 2.0 * b * (2 * i * h + 3 * h * h + 3 * h * o), 20)
    if kind == "vgg_front":
        b, px = case["batch"], float(case["height"] * case["width"])
        convs = [(3, 64, px), (64, 64, px), (64, 128, px / 4), (128, 128, px / 4)]
        flops = sum(18.0 * b * c * k * p * (2 if c == 3 else 3) for c, k, p in convs)
        return _training(sum(9 * c * k + k for c, k, _ in convs), b * px * (3 + 64 + 16 + 32 + 8), flops, 20)
    if kind in ("vgg16", "vgg16_eval"):
        b = case["batch"]
        convs = [(c, k, float(side * side)) for c, k, side in VGG_CONVS]
        if kind == "vgg16_eval":
            flops = sum(18.0 * b * c * k * p for c, k, p in convs) + sum(2.0 * b * i * o for i, o in VGG_LINEARS)
            images = float(b * case["minibatches"])
            return {"bytes": images * (3 * 224 * 224 * 4 + 4000) + 4.0 * VGG_PARAMS, "flops": case["minibatches"] * flops}
        flops = (sum(18.0 * b * c * k * p * (2 if c == 3 else 3) for c, k, p in convs)
                 + sum(6.0 * b * i * o for i, o in VGG_LINEARS))
        return _training(VGG_PARAMS, b * sum(c * p for c, _, p in convs) + b * sum(i for i, _ in VGG_LINEARS), flops, 20)
    if kind in ("gnmt", "gnmt_bidir"):
        rows, h, v = float(case["steps"] * case["batch"]), case["hidden"], case["vocab"]
        widths = [h] * 4 if kind == "gnmt" else [h, h, 2 * h, h, h, h]      # input width of every LSTM direction
        flops = sum(3 * 2.0 * rows * 4 * h * (w + h) for w in widths)
        params = sum(4 * h * (w + h) + 8 * h for w in widths)
        # gates, cell state and output of every layer; the embedding's table is updated whole
        return _training(params, rows * h * 6 * len(widths) + rows * h, flops, 28, v * h * (4 + 28))
    if kind == "gnmt_head":
        rows, h, v = float(case["steps"] * case["batch"]), case["hidden"], case["vocab"]
        return _training(h * v + v, rows * (h + v), 3 * 2.0 * rows * h * v, 28)
    if kind in ("transformer", "transformer_eval"):
        rows, s, h, n = float(case["batch"] * case["seq"]), case["seq"], case["hidden"], case["depth"]
        params, forward = n * (12.0 * h * h + 13 * h), n * (24.0 * rows * h * h + 4.0 * rows * s * h)
        if kind == "transformer_eval":
            return {"bytes": 2.0 * params + rows * h * 6, "flops": forward}
        m = _Transformer.MICRO_BATCHES
        # bf16: x, LN1, QKV, attention, x2, LN2 and the two hidden tensors of the feed-forward block per layer
        return {"bytes": m * (4.0 * n * rows * h * 16 + 4.0 * params + 16.0 * rows * h) + params * (4 + 28 + 2),
                "flops": m * 3.0 * forward}
    half = case["mixed"]
    per_param = {"sgd": 16, "adam": 24}[case["rule"]] + (2 + 2 if half else 4)
    return {"bytes": float(case["params"] * per_param), "flops": 0.0}


def tolerance(case):
    """About four times what the same step shows with its sums in another order (direct instead of Winograd
    convolutions, unsplit products on the fp32 matrix instructions, other bf16 tiles, unfused attention)."""
    return {
        # in a training step with ReLUs a few pre-activations lie within rounding of zero; whichever way they fall,
        # the gradients of that element's receptive field change
        "mlp": {"rel": 2e-3, "max": 0.1},
        "vgg_front": {"rel": 8e-3, "max": 0.2},
        "vgg16": {"rel": 3e-2, "max": 0.99},
        "vgg16_eval": {"rel": 1.5e-5},
        "gnmt": {"rel": 8e-6, "max": 3e-4},
        "gnmt_bidir": {"rel": 8e-6, "max": 3e-4},
        # (Adam's first steps take the sign of gradients that are all rounding)
        "gnmt_head": {"rel": 1.6e-5, "max": 2e-2},
        "transformer": {"rel": 2.5e-2, "max": 0.5},
        "transformer_eval": {"rel": 1e-2},         # bf16 activations
        "update": {"rel": 2e-6},
    }[case["kind"]]
