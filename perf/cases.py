"""The work that programs have minidist do on one MI355X, as cases to be timed and compared.

Four kinds of call, each through the package's public API over a ``ResidentGroup`` (W
data-parallel replicas on one GPU, the peers' contributions resident in its memory):

* ``ddp``   what follows a backward: ``finish_gradient_sync`` (pack x 1/W, W-way sum, unpack) and,
            with a loss scaler, ``unscale_`` and ``update``.  ``scaler`` says how the program uses it:
            ``fused`` (``DDP(..., grad_scaler=)``), ``own pass`` (the plain training loop) or ``none``.
* ``fsdp``  what an FSDP step moves besides the model's own arithmetic: the reduce-scatter of every
            unit's gradients into its fp32 shard, then the gather of its parameters.
* ``step``  a whole training step of a stack of linear layers under DDP, every bucket launched from
            the autograd hooks while backward goes on.
* ``coll``  the collectives by themselves: ``all_reduce`` in place, or a ``reduce_scatter_tensor``
            and an ``all_gather_into_tensor`` (a sharded optimizer's exchange).

Inputs come from the seed alone.  Gradients have the size a loss scale of 2^16 gives them where
there is a scaler.  A DDP program's gradients are tensors that autograd allocates, each 512-byte
aligned; here they are such slots of one buffer (``aligned``), or views packed one after another
from an odd element on (gradients that are views of a caller's own flat buffer).
"""

import math
import sys
from pathlib import Path

import torch
import torch.distributed as dist
from torch import nn

_PKG = str(Path(__file__).resolve().parent.parent / "distributed-training-framework_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_SIZES = {"f32": 4, "bf16": 2, "f16": 2}
_OPS = {"sum": dist.ReduceOp.SUM, "max": dist.ReduceOp.MAX, "min": dist.ReduceOp.MIN}
_SCALE = 2.0**16
_MAX_BYTES = 20e9  # of one drawn pass; the largest listed case moves 19.5 GB
_MAX_BUCKETS = 40


def listed():
    return [
        # The tiny GPT of the examples: one short dispatch, host latency counts.
        _gpt("ddp_tiny_gpt_f32_w4", 4, 256, 1024, 128, dtype="f32", world=4, rank=0, scaler="fused"),
        # GPT-2 124M in fp32 over 8 replicas, 25 MB buckets, fused loss scaler: the headline benchmark.
        _gpt("ddp_gpt2_f32_w8", 12, 768, 50257, 1024, dtype="f32", world=8, rank=0, scaler="fused"),
        # GPT-2 124M in fp16, the plain training loop: the scaler's unscale_ is a pass of its own.
        _gpt("ddp_gpt2_f16_w8_own_pass", 12, 768, 50257, 1024, dtype="f16", world=8, rank=3, scaler="own pass"),
        # GPT-2 medium in bf16 with buckets of its own dtype (the default), no scaler.
        _gpt("ddp_medium_bf16_w4", 24, 1024, 50257, 1024, dtype="bf16", world=4, rank=1, scaler="none"),
        # Four Llama-7B layers, bf16 gradients summed in fp32 buckets: the largest.
        dict(_LLAMA, name="ddp_llama_4l_bf16_f32_w8"),
        # An MLP of odd widths over 3 replicas, gradients as unaligned views: ragged everything.
        dict(kind="ddp", name="ddp_odd_mlp_f32_w3", model="mlp", layers=9, width=1531, vocab=0, ctx=0, dtype="f32",
             reduce="same", world=3, rank=2, scaler="fused", cap_mb=25.0, aligned=False),
        # One GPT-2 XL block as an FSDP unit (bf16 parameters, fp32 reduction): the per-unit exchange.
        dict(kind="fsdp", name="fsdp_xl_unit_bf16_w8", units=1, width=1600, param="bf16", reduce="f32", world=8, rank=0,
             accumulate=False),
        # GPT-2 sized blocks in fp16 over 6 ranks, gradients accumulated into the shards' own.
        dict(kind="fsdp", name="fsdp_gpt2_f16_w6_acc", units=12, width=768, param="f16", reduce="f32", world=6, rank=1,
             accumulate=True),
        # GPT-2 medium sized blocks with gradients reduced in bf16 as well.
        dict(kind="fsdp", name="fsdp_medium_bf16_reduce_w4", units=16, width=1024, param="bf16", reduce="bf16", world=4,
             rank=3, accumulate=False),
        # A training step with the buckets' launches inside backward.
        dict(kind="step", name="step_linear_bf16_w8", layers=8, width=4096, tokens=256, world=8, rank=0),
        # A few kilobytes summed in place: latency alone.
        dict(kind="coll", name="all_reduce_16kb_f32_w8", op="sum", numel=4096, dtype="f32", world=8, rank=0),
        # A sharded optimizer's exchange of 64M bf16 values.
        dict(kind="coll", name="rs_ag_64m_bf16_w8", op="rs_ag", numel=1 << 26, dtype="bf16", world=8, rank=5),
    ]


def _gpt(name, layers, width, vocab, ctx, **kw):
    case = dict(kind="ddp", name=name, model="gpt", layers=layers, width=width, vocab=vocab, ctx=ctx, reduce="same",
                cap_mb=25.0, aligned=True)
    case.update(kw)
    return case


_LLAMA = dict(kind="ddp", model="llama", layers=4, width=4096, vocab=0, ctx=11008, dtype="bf16", reduce="f32", world=8,
              rank=0, scaler="none", cap_mb=100.0, aligned=True)


def draw(rng):
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= _MAX_BYTES:
            return case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    world = rng.choice([2, 3, 4, 4, 5, 6, 7, 8, 8, 8, 12, 16])
    rank = rng.randrange(world)
    kind = rng.choice(["ddp", "ddp", "ddp", "fsdp", "fsdp", "coll", "coll", "step"])
    if kind == "ddp":
        dtype = rng.choice(["f32", "bf16", "f16"])
        case = dict(kind="ddp", model=rng.choice(["gpt", "gpt", "llama", "mlp"]), layers=rng.randint(2, 24),
                    width=_log(rng, 100, 2048), vocab=_log(rng, 500, 51000), ctx=_log(rng, 64, 2048), dtype=dtype,
                    reduce="f32" if dtype != "f32" and rng.random() < 0.5 else "same", world=world, rank=rank,
                    scaler=rng.choice(["fused", "own pass", "none"]), cap_mb=rng.choice([1.0, 25.0, 25.0, 100.0]),
                    aligned=rng.random() < 0.75)
        while len(_buckets(case)) > _MAX_BUCKETS:
            case["cap_mb"] *= 2
        return case
    if kind == "fsdp":
        param = rng.choice(["bf16", "bf16", "f16", "f32"])
        return dict(kind="fsdp", units=rng.choice([1, 1, 2, 4, 8, 16, 24]), width=_log(rng, 64, 1700), param=param,
                    reduce=rng.choice(["f32", "f32", param]), world=world, rank=rank, accumulate=rng.random() < 0.3)
    if kind == "step":
        return dict(kind="step", layers=rng.randint(2, 12), width=rng.choice([512, 1000, 1024, 2048, 2560, 4096]),
                    tokens=rng.choice([64, 200, 256, 512]), world=world, rank=rank)
    return dict(kind="coll", op=rng.choice(["sum", "sum", "max", "min", "rs_ag", "rs_ag"]), numel=_log(rng, 1, 1 << 28),
                dtype=rng.choice(["f32", "bf16", "f16"]), world=world, rank=rank)


# -- shapes ---------------------------------------------------------------------------------------


def _block_shapes(h):
    """A pre-norm GPT block: norm, qkv, projection, norm, two feed-forward layers (weight, bias each)."""
    return [(h,), (h,), (3 * h, h), (3 * h,), (h, h), (h,), (h,), (h,), (4 * h, h), (4 * h,), (h, 4 * h), (h,)]


def _shapes(case):
    h, layers = case["width"], case["layers"]
    if case["model"] == "gpt":
        return [(case["ctx"], h), (case["vocab"], h), *(s for _ in range(layers) for s in _block_shapes(h)), (h,), (h,)]
    if case["model"] == "llama":
        ffn = case["ctx"] if case["ctx"] > h else 3 * h
        layer = [(h,), (h, h), (h, h), (h, h), (h, h), (h,), (ffn, h), (ffn, h), (h, ffn)]
        return [s for _ in range(layers) for s in layer]
    return [s for i in range(layers) for s in ((h + 2 * i, h - 3 * i), (h + 2 * i,))]  # mlp


def _buckets(case):
    """Parameter indices of each bucket: reverse order, closed before the parameter that would pass the cap."""
    cap, out, filled = int(case["cap_mb"] * 2**20), [], 0
    for i, shape in reversed(list(enumerate(_shapes(case)))):
        n = math.prod(shape) * _SIZES[case["dtype"]]
        if not out or filled + n > cap:
            out.append([])
            filled = 0
        out[-1].append(i)
        filled += n
    return out


def _slots(shapes, esize, aligned):
    """Each gradient's first element in the gradient buffer, and the buffer's length."""
    starts, at, step = [], 0 if aligned else 1, 512 // esize
    for s in shapes:
        starts.append(at)
        at += math.prod(s)
        if aligned:
            at = -(-at // step) * step
    return starts, at


def _generator(seed):
    return torch.Generator("cuda").manual_seed(seed)


def _std(case):
    return 64.0 if case.get("scaler", "none") != "none" else 1e-3


# -- ddp ------------------------------------------------------------------------------------------


def _prepare_ddp(case, seed):
    from minidist import DDP, DistributedGradScaler, ResidentGroup

    gen, dtype, W = _generator(seed), _DTYPES[case["dtype"]], case["world"]
    shapes = _shapes(case)
    model = nn.Module()
    model.ps = nn.ParameterList([nn.Parameter(torch.zeros(s, dtype=dtype, device="cuda")) for s in shapes])
    group = ResidentGroup(W, case["rank"])
    scaler = DistributedGradScaler(init_scale=_SCALE, process_group=group) if case["scaler"] != "none" else None
    ddp = DDP(model, process_group=group, bucket_cap_mb=case["cap_mb"], broadcast_parameters=False,
              grad_scaler=scaler if case["scaler"] == "fused" else None,
              reduce_dtype=torch.float32 if case["reduce"] == "f32" else None)
    starts, length = _slots(shapes, _SIZES[case["dtype"]], case["aligned"])
    flat = torch.zeros(length, dtype=dtype, device="cuda")
    for p, a in zip(ddp.module.parameters(), starts):
        p.grad = flat[a : a + p.numel()].view(p.shape).normal_(0, _std(case), generator=gen)
    raw = case["reduce"] == "f32" and case["dtype"] != "f32"
    rows = []
    for k in range(len(_buckets(case))):
        replicas = ddp.bucket_replicas(k)
        rows.append(replicas[case["rank"]])
        for r in range(W):
            if r != case["rank"]:
                replicas[r].normal_(0, _std(case) / (1 if raw else W), generator=gen)
    opt = torch.optim.SGD(ddp.module.parameters(), lr=0.1)
    return dict(kind="ddp", ddp=ddp, scaler=scaler, opt=opt, flat=flat, rows=rows)


def _run_ddp(st):
    st["ddp"].finish_gradient_sync()
    out = {"grads": st["flat"], "rows": st["rows"]}
    if st["scaler"] is not None:
        out["found_inf"] = st["scaler"].unscale_(st["opt"])
        st["scaler"].update()
    return out


def _exact_ddp(case, seed):
    gen, dtype, W = _generator(seed), _DTYPES[case["dtype"]], case["world"]
    shapes = _shapes(case)
    starts, length = _slots(shapes, _SIZES[case["dtype"]], case["aligned"])
    flat = torch.zeros(length, dtype=dtype, device="cuda")
    for shape, a in zip(shapes, starts):
        flat[a : a + math.prod(shape)].normal_(0, _std(case), generator=gen)
    flat = flat.double()
    raw = case["reduce"] == "f32" and case["dtype"] != "f32"
    inv = 1.0 if case["scaler"] == "none" else 1.0 / _SCALE
    rows = []
    for members in _buckets(case):
        own = torch.cat([flat[starts[i] : starts[i] + math.prod(shapes[i])] for i in members])
        rows.append(own if raw else own / W)
        total = own / W
        for r in range(W):
            if r != case["rank"]:
                peer = torch.empty(own.numel(), dtype=dtype, device="cuda")
                peer.normal_(0, _std(case) / (1 if raw else W), generator=gen)
                total += peer.double() / (W if raw else 1)
        total *= inv
        at = 0
        for i in members:
            n = math.prod(shapes[i])
            flat[starts[i] : starts[i] + n] = total[at : at + n]
            at += n
    out = {"grads": flat, "rows": rows}
    if case["scaler"] != "none":
        out["found_inf"] = False
    return out


# -- fsdp -----------------------------------------------------------------------------------------


class _Block(nn.Module):
    def __init__(self, h):
        super().__init__()
        self.ps = nn.ParameterList([nn.Parameter(torch.zeros(s, device="cuda")) for s in _block_shapes(h)])


def _shard(case):
    """Elements of a unit, and of one rank's shard of it."""
    total = sum(math.prod(s) for s in _block_shapes(case["width"]))
    return total, -(-total // case["world"])


def _fsdp_inputs(case, gen, unit):
    """Fills one unit's tensors, in this order: the master shard, the peers' gathered shards, the
    peers' gradients, this rank's gradients and, where gradients accumulate, the shard's so far."""
    W, rank = case["world"], case["rank"]
    unit["master"].normal_(0, 0.02, generator=gen)
    for r in range(W):
        if r != rank:
            unit["peer_shards"][r].normal_(0, 0.02, generator=gen)
    for r in range(W):
        if r != rank:
            unit["peer_grads"][r].normal_(0, 1e-3, generator=gen)
    unit["grads"].normal_(0, 1e-3, generator=gen)
    if case["accumulate"]:
        unit["so_far"].normal_(0, 1e-3, generator=gen)


def _prepare_fsdp(case, seed):
    from minidist import FSDP, MixedPrecisionPolicy, ResidentGroup

    gen, param = _generator(seed), _DTYPES[case["param"]]
    total, S = _shard(case)
    root = nn.Module()
    root.blocks = nn.ModuleList([_Block(case["width"]) for _ in range(case["units"])])
    fsdp = FSDP(root, unit_types=(_Block,), process_group=ResidentGroup(case["world"], case["rank"]),
                mixed_precision=MixedPrecisionPolicy(param, _DTYPES[case["reduce"]]), broadcast_parameters=False,
                device=torch.device("cuda", torch.cuda.current_device()))
    shapes = _block_shapes(case["width"])
    starts, length = _slots(shapes, _SIZES[case["param"]], True)
    grads, shards, full = [], [], []
    for u in fsdp._units:
        t = dict(master=u.flat_shard.data, peer_shards=u.peer_param_shards(), peer_grads=u.peer_grad_contributions(),
                 grads=torch.empty(length, dtype=param, device="cuda"))
        if case["accumulate"]:
            t["so_far"] = u.flat_shard.grad = torch.empty(S, device="cuda")
        _fsdp_inputs(case, gen, t)
        grads += [(p, t["grads"][a : a + p.numel()].view(p.shape)) for p, a in zip(u.params, starts)]
        shards.append(u.flat_shard)
        full.append(u._full)  # the gathered parameters: finish_gradient_sync frees their storage, unshard fills it
    return dict(kind="fsdp", fsdp=fsdp, grads=grads, shards=shards, full=full, accumulate=case["accumulate"])


def _run_fsdp(st):
    for p, g in st["grads"]:  # what backward leaves
        p.grad = g
    if not st["accumulate"]:
        for s in st["shards"]:
            s.grad = None
    st["fsdp"].finish_gradient_sync()
    for u in st["fsdp"]._units:  # the next forward's gathers, one unit after another
        u.unshard()
    return {"shard_grads": [s.grad for s in st["shards"]], "params": st["full"]}


def _exact_fsdp(case, seed):
    gen, param, W, rank = _generator(seed), _DTYPES[case["param"]], case["world"], case["rank"]
    total, S = _shard(case)
    shapes = _block_shapes(case["width"])
    starts, length = _slots(shapes, _SIZES[case["param"]], True)
    out = {"shard_grads": [], "params": []}
    for _ in range(case["units"]):
        t = dict(master=torch.empty(S, device="cuda"), peer_shards=torch.empty(W, S, dtype=param, device="cuda"),
                 peer_grads=torch.zeros(W, S * W, dtype=param, device="cuda"),
                 grads=torch.empty(length, dtype=param, device="cuda"), so_far=torch.zeros(S, device="cuda"))
        _fsdp_inputs(case, gen, t)
        own = torch.zeros(S * W, dtype=torch.float64, device="cuda")
        at = 0
        for s, a in zip(shapes, starts):
            n = math.prod(s)
            own[at : at + n] = t["grads"][a : a + n]
            at += n
        mine = slice(rank * S, (rank + 1) * S)
        reduced = own[mine] / W
        for r in range(W):
            if r != rank:
                reduced += t["peer_grads"][r][mine].double() / W
        out["shard_grads"].append(reduced + t["so_far"].double())
        out["params"].append(torch.cat([(t["master"] if r == rank else t["peer_shards"][r]).double() for r in range(W)]))
    return out


# -- step -----------------------------------------------------------------------------------------


def _step_model(case, gen):
    h = case["width"]
    layers = [nn.Linear(h, h, device="cuda", dtype=torch.bfloat16) for _ in range(case["layers"])]
    for m in layers:
        m.weight.data.normal_(0, h**-0.5, generator=gen)
        m.bias.data.normal_(0, 0.02, generator=gen)
    x = torch.empty(case["tokens"], h, dtype=torch.bfloat16, device="cuda").normal_(generator=gen)
    return nn.Sequential(*layers), x


def _prepare_step(case, seed):
    from minidist import DDP, ResidentGroup

    gen, W, rank = _generator(seed), case["world"], case["rank"]
    model, x = _step_model(case, gen)
    ddp = DDP(model, process_group=ResidentGroup(W, rank), broadcast_parameters=False, reduce_dtype=torch.float32)
    # The peers' gradients, by parameter (the rows of a bucket hold its parameters one after another).
    peer = _step_peers(case, gen)
    k, row, at = 0, ddp.bucket_replicas(0), 0
    for i in reversed(range(2 * case["layers"])):
        n = peer[i].shape[1]
        if at == row[0].numel():
            k, at = k + 1, 0
            row = ddp.bucket_replicas(k)
        for r in range(W):
            if r != rank:
                row[r][at : at + n] = peer[i][r]
        at += n
    return dict(kind="step", ddp=ddp, x=x)


def _step_peers(case, gen):
    h, W = case["width"], case["world"]
    return [torch.empty(W, n, dtype=torch.bfloat16, device="cuda").normal_(0, 0.1, generator=gen)
            for _ in range(case["layers"]) for n in (h * h, h)]


def _run_step(st):
    for p in st["ddp"].module.parameters():
        p.grad = None
    out = st["ddp"](st["x"])
    out.backward(out.detach())  # the gradient of half the sum of squares
    return {"out": out.detach(), "grads": [p.grad for p in st["ddp"].module.parameters()]}


def _exact_step(case, seed):
    gen, W, rank = _generator(seed), case["world"], case["rank"]
    model, x = _step_model(case, gen)
    peers = _step_peers(case, gen)
    model = model.double()
    out = model(x.double())
    out.backward(out.detach())
    grads = []
    for p, peer in zip(model.parameters(), peers):
        total = p.grad.reshape(-1) / W
        for r in range(W):
            if r != rank:
                total += peer[r].double() / W
        grads.append(total.view(p.shape))
    return {"out": out.detach(), "grads": grads}


# -- coll -----------------------------------------------------------------------------------------


def _prepare_coll(case, seed):
    from minidist import ResidentGroup, comm

    gen, dtype, W, rank, n = _generator(seed), _DTYPES[case["dtype"]], case["world"], case["rank"], case["numel"]
    group = ResidentGroup(W, rank)
    if case["op"] != "rs_ag":
        row = group.zeros(n, dtype)
        for t in group.replicas(row):
            t.normal_(generator=gen)
        return dict(kind="coll", comm=comm, group=group, row=row, op=_OPS[case["op"]])
    S = -(-n // W)
    grads, shard = group.zeros(S * W, dtype), group.zeros(S, dtype)
    for t in (*group.replicas(grads), *group.replicas(shard)):
        t.normal_(generator=gen)
    return dict(kind="coll", comm=comm, group=group, grads=grads, shard=shard, op=None,
                mine=torch.empty(S, dtype=dtype, device="cuda"), full=torch.empty(S * W, dtype=dtype, device="cuda"))


def _run_coll(st):
    comm, group = st["comm"], st["group"]
    if st["op"] is not None:
        comm.all_reduce(st["row"], op=st["op"], group=group)
        return st["row"]
    comm.reduce_scatter_tensor(st["mine"], st["grads"], group=group)
    comm.all_gather_into_tensor(st["full"], st["shard"], group=group)
    return {"mine": st["mine"], "full": st["full"]}


def _exact_coll(case, seed):
    gen, dtype, W, rank, n = _generator(seed), _DTYPES[case["dtype"]], case["world"], case["rank"], case["numel"]

    def rows(m):
        for _ in range(W):
            yield torch.empty(m, dtype=dtype, device="cuda").normal_(generator=gen).double()

    if case["op"] != "rs_ag":
        fold = {"sum": torch.add, "max": torch.maximum, "min": torch.minimum}[case["op"]]
        acc = None
        for t in rows(n):
            acc = t if acc is None else fold(acc, t)
        return acc
    S = -(-n // W)
    mine = sum(t[rank * S : (rank + 1) * S] for t in rows(S * W))
    return {"mine": mine, "full": torch.cat(list(rows(S)))}


# -- the whole ------------------------------------------------------------------------------------


def prepare(case, seed):
    return {"ddp": _prepare_ddp, "fsdp": _prepare_fsdp, "step": _prepare_step, "coll": _prepare_coll}[case["kind"]](case, seed)


def run(state):
    return {"ddp": _run_ddp, "fsdp": _run_fsdp, "step": _run_step, "coll": _run_coll}[state["kind"]](state)


def exact(case, seed):
    return {"ddp": _exact_ddp, "fsdp": _exact_fsdp, "step": _exact_step, "coll": _exact_coll}[case["kind"]](case, seed)


def work(case):
    """Bytes: each contribution read once, each result written once (ddp: the gradient and the peers' rows in; the
    packed row, the bucket and the gradient out; a scaler's pass of its own adds none that a fused one would not need)."""
    W = case["world"]
    if case["kind"] == "ddp":
        n, es = sum(math.prod(s) for s in _shapes(case)), _SIZES[case["dtype"]]
        bucket = 4 if case["reduce"] == "f32" else es
        return {"bytes": n * ((W + 2) * es + bucket), "flops": 0}
    if case["kind"] == "fsdp":
        (total, S), es = _shard(case), _SIZES[case["param"]]
        reduce = S * (W * es + 4 + (4 if case["accumulate"] else 0))
        gather = S * (4 + es) + 2 * (W - 1) * S * es
        return {"bytes": case["units"] * (reduce + gather), "flops": 0}
    if case["kind"] == "step":
        h, L, T = case["width"], case["layers"], case["tokens"]
        n = L * (h * h + h)
        # weights read forward and backward, gradients written once by backward; activations in and out of each product
        model = 2 * (3 * n + L * 6 * T * h)
        return {"bytes": model + n * ((W + 2) * 2 + 4), "flops": L * 6 * T * h * h}
    es, n = _SIZES[case["dtype"]], case["numel"]
    if case["op"] != "rs_ag":
        return {"bytes": n * (W + 1) * es, "flops": 0}
    S = -(-n // W)
    return {"bytes": (W + 1) * S * es + 2 * W * S * es, "flops": 0}


def tolerance(case):
    """About four times the relative error seen against 64 bits: of a sum of W terms in the dtype it is taken in, or
    of the one rounding to 16 bits where the sum is taken in fp32.  Maxima and minima are values of the inputs."""
    if case["kind"] == "step":
        return {"rel": 2e-2}  # bf16 products, activations and gradients
    if case["kind"] == "coll" and case["op"] in ("max", "min"):
        return "exact"
    dtype = case["param"] if case["kind"] == "fsdp" else case["dtype"]
    if case.get("reduce") == "f32" and dtype != "f32":
        return {"rel": {"f16": 1e-3, "bf16": 7e-3}[dtype]}
    return {"rel": {"f32": 4e-7, "f16": 2e-3, "bf16": 1.6e-2}[dtype]}
