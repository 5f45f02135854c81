"""What the speed of this framework is judged on: whole passes of compiled programs, as a program that serves them
runs them.

Sizes come from the benchmark's workloads (bench.py), the tests and the graph builders (occamy_amd/models.py);
`draw` spreads them over the ranges around those: batches from one image to the largest that the benchmark runs,
image sides that are no multiple of anything, sequences of any length.  A program is compiled once and its session
(weights on the device, plan, recorded launches) kept for as long as inputs keep coming, which is what
`_session` does for the states of one case; a state holds the input and result buffers of one request.
"""
import functools

import numpy as np
import torch

from occamy_amd import compiler, models

_DTYPES = {"f32": (np.float32, torch.float32), "f16": (np.float16, torch.float16)}

# the compile flags of bench.py's workloads, by model
_RESNET = dict(fusion=True, fuse_residual=True, fuse_matmul_bias=True, fuse_first_layer_maxpool=True,
               fuse_projection_shortcut=True, alias_copies=True)
_IN_PLACE = dict(inplace_residual=True, compact_pool=True)
_BERT = dict(recompose=True, fusion=True, fuse_matmul_bias=True, fuse_attention=True, alias_copies=True)


def listed():
    return [
        # the smallest call: one 3x3 convolution block with bias and ReLU, launched for one image; launch and host time
        _conv_block("conv_block_f32_b1", "f32", 1, 64, 64, 56, 56, 3, 1),
        # interactive inference, one image or sentence at a time, in the reference's own type
        _image("resnet50_f32_b1", "resnet50", "f32", 1, 224, 224),
        _image("mobilenet_v2_f32_b1", "mobilenet_v2", "f32", 1, 224, 224),
        _bert("bert_f32_s128", "f32", 12, 128),
        # the call the reference's generated code makes: host arrays in and out, pool and weights set up per inference
        dict(_image("resnet50_f32_b1_host", "resnet50", "f32", 1, 224, 224), host=True),
        # batched classification in the reference's type
        _image("resnet50_f32_b32", "resnet50", "f32", 32, 224, 224),
        # throughput serving in half precision
        _image("resnet50_f16_b64", "resnet50", "f16", 64, 224, 224),
        _image("mobilenet_v2_f16_b64", "mobilenet_v2", "f16", 64, 224, 224),
        _bert("bert_f16_s384", "f16", 12, 384),
        # detection: large 3x3 layers and 25-million-weight classifiers; feature maps of 38, 19, 10, 5, 3 and 1 pixels
        _image("yolo_v1_f32_b2", "yolo_v1", "f32", 2, 448, 448),
        _image("ssd_resnet50_f32_b3", "ssd_resnet50", "f32", 3, 300, 300),
        # super-resolution of an image as it comes: sides of no particular size
        _image("srgan_f32_90x117", "srgan", "f32", 1, 90, 117),
    ]


def _conv_block(name, dtype, batch, cin, cout, height, width, kernel, stride):
    return {"name": name, "model": "conv_block", "dtype": dtype, "batch": batch, "cin": cin, "cout": cout, "height": height,
            "width": width, "kernel": kernel, "stride": stride, "host": False}


def _image(name, model, dtype, batch, height, width):
    return {"name": name, "model": model, "dtype": dtype, "batch": batch, "height": height, "width": width, "host": False}


def _bert(name, dtype, layers, seq):
    return {"name": name, "model": "bert", "dtype": dtype, "batch": 1, "layers": layers, "seq": seq, "host": False}


def draw(rng):
    while True:
        c = _draw(rng)
        if all(_key(c) != _key(x) for x in listed()):
            return c


def _draw(rng):
    def log(lo, hi):  # a whole number from lo to hi, spread over its logarithm
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["conv_block", "resnet50_f32", "resnet50_f16", "resnet50_host", "mobilenet_v2_f32", "mobilenet_v2_f16", "bert_f32",
                       "bert_f16", "yolo_v1", "ssd_resnet50", "srgan", "alexnet"])
    if kind == "conv_block":
        cin, cout = (rng.choice([16, 24, 32, 48, 64, 96, 128, 192, 256]) for _ in range(2))
        side = log(7, 112)
        c = _conv_block("", "f32", rng.choice([1, 1, 2, 4]), cin, cout, side, max(7, side - rng.randrange(0, 5)), rng.choice([1, 3, 3, 5]), rng.choice([1, 1, 2]))
    elif kind in ("resnet50_f32", "resnet50_f16", "mobilenet_v2_f32", "mobilenet_v2_f16"):
        side = rng.randrange(128, 289)
        most = (32 if kind == "resnet50_f32" else 64) * 224 * 224 // (side * side)
        c = _image("", kind[:-4], kind[-3:], min(log(1, 64), most), side, side)
    elif kind == "resnet50_host":
        side = rng.randrange(128, 289)
        c = dict(_image("", rng.choice(["resnet50", "mobilenet_v2"]), "f32", log(1, 8), side, side), host=True)
    elif kind in ("bert_f32", "bert_f16"):
        c = _bert("", kind[-3:], rng.choice([2, 4, 6, 12]), log(16, 512))
    elif kind == "yolo_v1":
        side = 64 * rng.randrange(3, 9)
        c = _image("", "yolo_v1", "f32", rng.randrange(1, 5), side, side)
    elif kind == "ssd_resnet50":
        c = _image("", "ssd_resnet50", "f32", rng.randrange(1, 4), 300, 300)
        c["height"] = c["width"] = rng.randrange(288, 313)
    elif kind == "srgan":
        c = _image("", "srgan", "f32", rng.randrange(1, 3), log(16, 128), log(16, 128))
    else:
        c = _image("", "alexnet", "f32", log(1, 32), 224, 224)
    del c["name"]
    return c


def _graph(case):
    """The case's graph and compile flags."""
    m, dt, batch = case["model"], _DTYPES[case["dtype"]][0], case["batch"]
    half = dict(channels_last=True) if case["dtype"] == "f16" else {}
    if m == "conv_block":
        g = compiler.Graph()
        r = np.random.default_rng(1)
        k, cin, cout = case["kernel"], case["cin"], case["cout"]
        bound = float(np.sqrt(6.0 / (cin * k * k)))
        x = g.input("X", (batch, cin, case["height"], case["width"]), dt)
        w = g.constant(r.uniform(-bound, bound, (cout, cin, k, k)).astype(dt))
        b = g.constant(r.uniform(-0.1, 0.1, (cout,)).astype(dt))
        c = g.node("Conv", [x, w, b], kernel_shape=[k, k], pads=[k // 2] * 4, strides=[case["stride"]] * 2, group=1)
        g.output(g.node("Relu", [c]))
        return g, dict(fusion=True)
    if m == "resnet50":
        flags = dict(fusion=True) if case["host"] else dict(_RESNET, **half, **(_IN_PLACE if batch > 1 else {}))
        return models.resnet50(batch, dt, image=case["height"])[0], flags
    if m == "mobilenet_v2":
        flags = dict(fusion=True, fuse_residual=True, fuse_activations=True, fuse_matmul_bias=True, alias_copies=True, **half, **(_IN_PLACE if batch > 1 else {}))
        return models.mobilenet_v2(batch, dt, image=case["height"])[0], dict(fusion=True) if case["host"] else flags
    if m == "bert":
        return models.bert_encoder(layers=case["layers"], seq=case["seq"], dtype=dt)[0], dict(_BERT, **(dict(compact_pool=True) if half else {}))
    if m == "yolo_v1":
        return models.yolo_v1(batch, dt, image=case["height"])[0], dict(fusion=True, fuse_activations=True, fuse_matmul_bias=True)
    if m == "ssd_resnet50":
        flags = dict(fusion=True, fuse_residual=True, fuse_first_layer_maxpool=True, fuse_projection_shortcut=True, **_IN_PLACE)
        return models.ssd_resnet50(batch, dt, image=case["height"])[0], flags
    if m == "srgan":
        return models.srgan_generator(batch, dt, height=case["height"], width=case["width"])[0], dict(fusion=True, fuse_residual=True, fuse_activations=True)
    return models.alexnet(batch, dt, image=case["height"])[0], dict(fusion=True, fuse_matmul_bias=True)


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


@functools.lru_cache(maxsize=16)
def _program(key):
    graph, flags = _graph(dict(key))
    return graph, graph.compile(**flags)


@functools.lru_cache(maxsize=16)
def _session(key):
    _, program = _program(key)
    return program.session(compiler.MODE_OCCAMY if dict(key)["host"] else compiler.MODE_RESIDENT)


def prepare(case, seed):
    graph, program = _program(_key(case))
    (shape, dtype), = graph.input_shapes.values()
    r = torch.Generator(device="cpu" if case["host"] else "cuda").manual_seed(seed)
    if dtype == np.int64:  # token ids
        x = torch.randint(0, 30522, shape, generator=r, device=r.device)
    else:  # a normalised image or feature map
        x = torch.randn(shape, generator=r, device=r.device).to(_DTYPES[case["dtype"]][1])
    state = {"session": _session(_key(case))}
    if case["host"]:
        return dict(state, x=x.numpy())
    out = [torch.empty(s, dtype=_DTYPES[case["dtype"]][1], device="cuda") for s, _ in program.output_info()]
    torch.cuda.synchronize()  # the session has a stream of its own
    return dict(state, x=x, out=out, inputs=[x.data_ptr()], outputs=[t.data_ptr() for t in out])


def run(state):
    if "out" not in state:
        return state["session"].run(state["x"])
    state["session"].run_device(state["inputs"], state["outputs"], use_graph=True, in_place=True)
    return state["out"]


def work(case):
    """Operations: those of the convolutions, products and everything between them.  Bytes: weights, input and results,
    each once (of an embedding table the rows that are looked up); what lies between layers need not leave the chip."""
    graph, program = _program(_key(case))
    size = np.dtype(_DTYPES[case["dtype"]][0]).itemsize
    (shape, dtype), = graph.input_shapes.values()
    total = int(np.prod(shape)) * np.dtype(dtype).itemsize + sum(int(np.prod(s)) * np.dtype(d).itemsize for s, d in program.output_info())
    for name, a in graph.constants.items():
        if a.dtype != np.int64:
            total += min(a.size, case["seq"] * a.shape[1]) * size if name == "word_embeddings" else a.nbytes
    return {"bytes": total, "flops": sum(op[2] for op in program.compute_ops())}


def tolerance(case):
    """fp32 sums in another order, through up to fifty layers; fp16: every layer's result is rounded to 11 bits."""
    return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 5e-3}
