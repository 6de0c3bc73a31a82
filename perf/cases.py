"""The calls that the chains' speed is judged by: what a program built on this package has it do, over the range it
does it in.

Every case goes through a public entry point: a function that ``ditto_amd.build`` returned (``entry`` "built", and
"conv" with its weights bound by ``specialize``), ``chain.run_bmm_chain`` on the caller's tensors ("tensors"), the
attention module on a packed projection ("packed"), or a stack of attention layers in the graph-replay engine
("layers").  Shapes are those of the drivers' tables (``ditto_amd/drivers/common.py``), of ``bench.py`` and of the
tests, at batch sizes from one upwards; ``draw`` spreads sizes over the same ranges, ragged ones among them.
"""
import math

import torch

import ditto_amd as ditto
from ditto_amd import auto_compute as ac
from ditto_amd import auto_schedule, chain, chimera, runtime
from ditto_amd.drivers import common

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32, "int8": torch.int8}
BYTES = {"float16": 2, "bfloat16": 2, "float32": 4, "int8": 1}

# no drawn case does more than this
MAX_FLOPS = {"built": 5.5e11, "tensors": 5.5e11, "packed": 5.5e11, "layers": 1.2e11, "conv": 3.1e10}
MAX_FLOPS_F32 = 2.5e9
MAX_BYTES = 2.7e8


def listed():
    return [
        # the first layer of a small MLP-Mixer (drivers' table): a call as short as they come
        dict(name="gemm_f16_mixer", entry="built", dtype="float16", inter="cast", batch=1, M=512, L=256, D=64),
        # a BERT-base encoder's attention at batch 8 and full length, twelve layers replayed as one graph
        dict(name="bert_layers_f16", entry="layers", dtype="float16", layers=12, batch=8, M=512, heads=12, D=64),
        # ViT-Huge attention (heads of 80) on a packed projection; 196 patches and the class token make 197 rows
        dict(name="vit_packed_bf16", entry="packed", dtype="bfloat16", batch=16, M=197, heads=16, D=80),
        # long-sequence attention: the benchmark's headline, the largest call
        dict(name="attn_bf16_long", entry="tensors", dtype="bfloat16", inter="softmax", batch=64, M=4096, L=4096, D=128),
        # the large GEMM chain, B as the operator builders lay it out
        dict(name="gemm_bf16_large", entry="built", dtype="bfloat16", inter="cast", batch=64, M=4096, L=4096, D=128),
        # quantised MLP: int8 in, middle result requantised per column, int32 out
        dict(name="gemm_i8_requant", entry="built", dtype="int8", inter="requant", batch=1, M=8192, K=1024, L=256, N=1024),
        # single precision attention of BERT-base size at batch 1 (the CPU-sized configurations' data type)
        dict(name="attn_f32_bert", entry="tensors", dtype="float32", inter="softmax", batch=12, M=512, L=512, D=64),
        # ResNet bottleneck tail at batch 32
        dict(name="conv331_resnet", entry="conv", dtype="float16", relu=False, groups=False, N=32, C0=64, H=56, C1=64, R1=3,
             stride=1, C2=256, R2=1),
        # Inception stem: strided, image rows of odd length, channels that fill no tile
        dict(name="conv331_inception", entry="conv", dtype="float16", relu=True, groups=False, N=8, C0=32, H=147, C1=64,
             R1=3, stride=2, C2=80, R2=1),
        # Darknet block on one image: wide filters, few pixels
        dict(name="conv331_darknet_1", entry="conv", dtype="float16", relu=False, groups=False, N=1, C0=128, H=28, C1=256,
             R1=3, stride=1, C2=128, R2=1),
        # ResNet bottleneck head at batch 32
        dict(name="conv133_resnet", entry="conv", dtype="bfloat16", relu=True, groups=False, N=32, C0=64, H=56, C1=64, R1=1,
             stride=1, C2=64, R2=3),
        # depthwise-separable block of MobileNet with the drivers' channel multiplier of 16
        dict(name="dw_mobilenet", entry="conv", dtype="float16", relu=False, groups=True, N=32, C0=32, H=112, C1=512, R1=3,
             stride=1, C2=64, R2=1),
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, int(round(v / step)) * step)


# (C0, C1, C2, R1, R2, stride, depthwise): the drivers' convolution rows, a ResNet tail and multiplier-1 depthwise rows
_CONV_ROWS = [
    (64, 192, 128, 3, 1, 2, False), (32, 64, 80, 3, 1, 2, False), (64, 128, 64, 3, 1, 1, False),
    (128, 256, 128, 3, 1, 1, False), (16, 64, 16, 3, 1, 4, False), (64, 64, 256, 3, 1, 1, False),
    (64, 64, 64, 1, 3, 1, False), (64, 64, 64, 1, 3, 1, False), (64, 64, 64, 1, 1, 1, False),
    (256, 256, 64, 1, 1, 1, False), (32, 512, 64, 3, 1, 1, True), (32, 32, 64, 3, 1, 1, True),
    (64, 1024, 64, 3, 1, 1, True), (64, 64, 64, 3, 1, 1, True), (16, 256, 32, 3, 1, 2, True),
]


def draw(rng):
    entry = rng.choice(["built", "tensors", "packed", "layers", "int8", "float32", "conv", "conv", "conv"])
    half = rng.choice(["float16", "bfloat16"])
    if entry == "built":
        c = dict(entry="built", dtype=half, inter=rng.choice(["cast", "relu", "softmax"]), batch=_log_int(rng, 1, 64),
                 M=_log_int(rng, 128, 4096, 16), L=_log_int(rng, 64, 4096, 16), D=rng.choice([64, 80, 128]))
    elif entry == "tensors":  # attention: keys as stored, any number of rows
        m = _log_int(rng, 49, 4096)
        c = dict(entry="tensors", dtype=half, inter="softmax", batch=_log_int(rng, 1, 96), M=m,
                 L=m if rng.random() < 0.7 else _log_int(rng, 49, 4096), D=rng.choice([64, 80, 128]))
    elif entry == "packed":
        heads, d = rng.choice([(8, 64), (12, 64), (16, 64), (16, 80)])
        c = dict(entry="packed", dtype=half, batch=_log_int(rng, 1, 32), M=_log_int(rng, 49, 1024), heads=heads, D=d)
    elif entry == "layers":
        c = dict(entry="layers", dtype=half, layers=12, batch=_log_int(rng, 1, 8), M=_log_int(rng, 49, 512),
                 heads=rng.choice([8, 12, 16]), D=64)
    elif entry == "int8":
        c = dict(entry="built", dtype="int8", inter=rng.choice(["requant", "requant", "cast"]), batch=1,
                 M=_log_int(rng, 256, 8192, 16), K=_log_int(rng, 64, 1024, 16), L=_log_int(rng, 64, 512, 16),
                 N=_log_int(rng, 64, 1024, 16))
    elif entry == "float32":
        c = dict(entry="tensors", dtype="float32", inter=rng.choice(["softmax", "softmax", "cast"]),
                 batch=_log_int(rng, 1, 16), M=_log_int(rng, 49, 1024), L=_log_int(rng, 49, 1024), D=rng.choice([64, 80, 128]))
    else:
        C0, C1, C2, R1, R2, stride, groups = rng.choice(_CONV_ROWS)
        c = dict(entry="conv", dtype=half, relu=rng.random() < 0.5, groups=groups, N=_log_int(rng, 1, 32), C0=C0,
                 H=_log_int(rng, 17 * stride, 227 if stride > 1 else 112), C1=C1, R1=R1, stride=stride, C2=C2, R2=R2)
        if rng.random() < 0.5:  # the feature maps of image networks are mostly multiples of 28
            c["H"] = rng.choice([28, 56, 112] if stride == 1 else [112, 224])
    shrink = "N" if c["entry"] == "conv" else "batch"
    most = MAX_FLOPS_F32 if c["dtype"] == "float32" else MAX_FLOPS[c["entry"]]
    while c[shrink] > 1 and (work(c)["flops"] > most or work(c)["bytes"] > MAX_BYTES):
        c[shrink] = c[shrink] // 2
    return c


def _sizes(c):
    """(batch, M, K, L, N) of a chain of matrix products."""
    if c["entry"] in ("packed", "layers"):
        return c["batch"] * c["heads"], c["M"], c["D"], c["M"], c["D"]
    return c["batch"], c["M"], c.get("K", c.get("D")), c["L"], c.get("N", c.get("D"))


def _conv_out(c):
    """Output extent: the first filter is padded to keep the extent, the second one too."""
    p = (c["H"] + 2 * (c["R1"] // 2) - c["R1"]) // c["stride"] + 1
    return p


def work(case):
    c = case
    e = BYTES[c["dtype"]]
    if c["entry"] == "conv":
        p = _conv_out(c)
        c0 = 1 if c["groups"] else c["C0"]
        per_pixel = c["C1"] * c0 * c["R1"] ** 2 + c["C1"] * c["C2"] * c["R2"] ** 2
        values = (c["N"] * c["C0"] * c["H"] ** 2 + c["C1"] * c0 * c["R1"] ** 2 + c["C2"] * c["C1"] * c["R2"] ** 2
                  + c["N"] * c["C2"] * p * p)
        return {"bytes": e * values, "flops": 2.0 * c["N"] * p * p * per_pixel}
    b, m, k, l, n = _sizes(c)
    times = c.get("layers", 1)
    values = e * b * (m * k + k * l + l * n)
    out = b * m * n * (4 if c.get("inter") == "requant" else e)
    return {"bytes": times * (values + out), "flops": times * 2.0 * b * m * l * (k + n)}


def tolerance(case):
    if case["dtype"] == "int8":
        return "exact"
    # fp32 sums in another order; one rounding of the middle result and one of the output in the 16-bit types
    return {"rel": {"float32": 1e-5, "float16": 1e-3, "bfloat16": 6e-3}[case["dtype"]]}


def _normal(gen, shape, dtype, std=1.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _build(ins, outs, weights=0):
    split = len(ins) - weights
    layer = ac.layer([outs[0].op], inputs=ins[:split], weights=ins[split:])
    return ditto.build(common.describe_layer(layer), layer.schedule_tensors, "hip")


def _prepare_conv(c, gen):
    dt = DTYPES[c["dtype"]]
    p1, p2 = c["R1"] // 2, c["R2"] // 2
    ins, outs = ac.nn.functional.conv_chain(
        c["N"], c["C0"], c["H"], c["H"], c["C1"], c["R1"], c["R1"], c["C2"], c["R2"], c["R2"], p1, p2, c["stride"], 1,
        c["dtype"], "float32", relu=c["relu"], groups1=c["C0"] if c["groups"] else 1)
    x, w1, w2 = (_normal(gen, t.shape, dt, s) for t, s in
                 zip(ins, (1.0, (ins[1].shape[1] * c["R1"] ** 2) ** -0.5, (c["C1"] * c["R2"] ** 2) ** -0.5)))
    y = torch.empty(outs[0].shape, dtype=dt, device="cuda")
    return _build(ins, outs, weights=2).specialize(w1, w2), (x, w1, w2, y)


def _prepare_built(c, gen):
    b, m, k, l, n = _sizes(c)
    f = ac.nn.functional
    if c["dtype"] == "int8":
        ins, outs = f.BatchGemmGemm(b, m, n, k, l, "int8", "int32", scale_tensor=c["inter"] == "requant")
        args = [torch.randint(-127, 128, t.shape, dtype=torch.int8, device="cuda", generator=gen) for t in ins[:3]]
        if c["inter"] == "requant":
            # scales around the one that brings the middle result's spread to a third of the int8 range
            s = 40.0 / (5400.0 * k ** 0.5)
            args.append(s * (0.5 + torch.rand(l, device="cuda", generator=gen)))
        out = torch.empty((b, m, n), dtype=torch.int32 if c["inter"] == "requant" else torch.int8, device="cuda")
    else:
        dt = DTYPES[c["dtype"]]
        if c["inter"] == "softmax":
            ins, outs = f.BatchGemmSoftmaxGemm(b, m, n, k, l, c["dtype"], "float32", scale=k ** -0.5)
            std = (1.0, 1.0, 1.0)
        else:
            ins, outs = f.BatchGemmGemm(b, m, n, k, l, c["dtype"], "float32", relu=c["inter"] == "relu")
            std = (1.0, k ** -0.5, l ** -0.5)
        args = [_normal(gen, t.shape, dt, s) for t, s in zip(ins, std)]
        out = torch.empty((b, m, n), dtype=dt, device="cuda")
    return _build(ins, outs), (*args, out)


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[c["dtype"]]
    if c["entry"] == "conv":
        fn, args = _prepare_conv(c, gen)
    elif c["entry"] == "built":
        fn, args = _prepare_built(c, gen)
    elif c["entry"] == "tensors":
        b, m, k, l, n = _sizes(c)
        std = (1.0, 1.0, 1.0) if c["inter"] == "softmax" else (1.0, k ** -0.5, l ** -0.5)
        # keys and values as attention callers store them, one row per key
        q, key, v = (_normal(gen, s, dt, sd) for s, sd in zip(((b, m, k), (b, l, k), (b, l, n)), std))
        fn, args = chain.run_bmm_chain, (q, key.transpose(1, 2), v, torch.empty((b, m, n), dtype=dt, device="cuda"))
    else:
        mha = ac.nn.module.MultiHeadAttentionMMA(c["heads"], c["heads"] * c["D"], c["dtype"], "float32", scale=None)
        shape = (c["batch"], c["M"], 3 * c["heads"] * c["D"])
        if c["entry"] == "packed":
            fn, args = mha, (_normal(gen, shape, dt),)
        else:
            layers = [mha.layer(c["batch"], c["M"]) for _ in range(c["layers"])]
            graph = runtime.Graph(layers, outputs=[(i, 0) for i in range(c["layers"])])
            tasks = chimera.task_binding(auto_schedule.extract_tasks_from_graph(graph))
            option = auto_schedule.ScheduleOption("hip", log_file="untuned.log", dtype=c["dtype"])
            schedules = auto_schedule.retrieve_schedule_bound_tasks(tasks, option)
            built = {key: ditto.build(sch, tensors, "hip") for key, (sch, tensors) in schedules.items()}
            fn = runtime.create_hip_graph_engine(graph, built, "cuda:0")
            fn.set_inputs([_normal(gen, shape, dt) for _ in layers])
            fn.compile()
            args = ()
    return dict(c, fn=fn, args=args)


def run(state):
    fn, args = state["fn"], state["args"]
    if state["entry"] == "packed":
        return fn(*args)
    if state["entry"] == "layers":
        fn.run()
        return fn.get_outputs()
    if state["entry"] == "tensors":
        scale = state["D"] ** -0.5 if state["inter"] == "softmax" else 1.0
        return fn(*args, inter_op=state["inter"], softmax_scale=scale)
    fn(*args)
    return args[-1]
