"""The work whose time counts for users of this framework: cases that a measuring program prepares, runs and compares.

Six kinds of work, each over the range of sizes that it is used at:

  request  one scoring request of a CTR model through a Predictor: feed every input from host memory, forward, read the
           probabilities back (what a serving thread does per request)
  din      the same for a DIN-style model: attention over each sample's behaviour history
  serve    many forward passes of a CTR model by the library's serving threads, inputs resident on the device
  pool     one Embedding invocation at the kernel layer: gather and pool the ids of every slot
  fc       a tower of FC layers at the kernel layer: bias and activation per layer, a skinny head at the end
  bmm      a strided batched matrix product (MatMul over a batch: attention scores and weighted sums)
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "x-deeplearning_amd"))

import blaze_hip as bz  # noqa: E402
import ctr_model  # noqa: E402
import din_model  # noqa: E402
import pyblaze_hip as pb  # noqa: E402

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8}
SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1}
UDF = {"sum": bz.SUM, "avg": bz.AVG, "assign": bz.ASSIGN}
SERVING_THREADS = 8


def listed():
    return [
        # one sample at a time: the latency of the smallest request (the smallest benchmark model, fp32 throughout)
        dict(name="request_f32_one_sample", kind="request", dtype="f32", batch=1, slots=10, rows=1_000_000, dim=16, mean_len=5.5,
             zipf=1.1, keyed=False, dense=32, h1=200, h2=80),
        # re-ranking a few hundred candidates on tables that are looked up by key, as a trained model's are
        dict(name="request_f16_keyed_300", kind="request", dtype="f16", batch=300, slots=18, rows=100_000, dim=24, mean_len=3.0,
             zipf=1.1, keyed=True, dense=13, h1=256, h2=100),
        # the headline model and batch, every input crossing from host memory
        dict(name="request_f16_2048", kind="request", dtype="f16", batch=2048, slots=26, rows=1_000_000, dim=32, mean_len=8.0,
             zipf=1.1, keyed=False, dense=64, h1=512, h2=256),
        # attention over a short history in fp32, the reference's default type, at an odd batch
        dict(name="din_f32_201", kind="din", dtype="f32", batch=201, hist=23, rows=500_000, dim=16, zipf=1.2),
        # the attention model at its benchmark size
        dict(name="din_f16_1024", kind="din", dtype="f16", batch=1024, hist=50, rows=2_000_000, dim=18, zipf=1.2),
        # the headline throughput: eight serving threads, inputs resident
        dict(name="serve_f16_2048", kind="serve", dtype="f16", batch=2048, slots=26, rows=1_000_000, dim=32, mean_len=8.0,
             zipf=1.1, keyed=False, dense=64, h1=512, h2=256, predictors=16, passes=64),
        # fp32 tables looked up by key, odd dim, a batch that fills no whole number of workgroups
        dict(name="pool_f32_keyed_1000", kind="pool", dtype="f32", out="f32", batch=1000, slots=24, tables=4, rows=250_000,
             dim=100, mean_len=6.0, zipf=1.1, keyed=True, udf="sum", trunc=0),
        # quantised tables, long lists, mean pooling
        dict(name="pool_i8_avg_4096", kind="pool", dtype="i8", out="f16", batch=4096, slots=50, tables=50, rows=1_000_000, dim=64,
             mean_len=20.0, zipf=1.05, keyed=False, udf="avg", trunc=0),
        # the largest lookup: 200 slots of short lists over tables with no hot rows
        dict(name="pool_f16_200_slots", kind="pool", dtype="f16", out="bf16", batch=8192, slots=200, tables=200, rows=1_000_000,
             dim=64, mean_len=2.5, zipf=0.0, keyed=False, udf="sum", trunc=0),
        # the headline tower in fp32
        dict(name="fc_f32_2048", kind="fc", dtype="f32", batch=2048, k=896, h1=512, h2=256, h3=0, n=2, act="prelu"),
        # the largest tower: a wide first layer in bf16
        dict(name="fc_bf16_8192", kind="fc", dtype="bf16", batch=8192, k=12800, h1=1024, h2=512, h3=256, n=1, act="relu"),
        # attention scores q * k^T of every sample
        dict(name="bmm_f16_scores", kind="bmm", dtype="f16", batch=1024, m=50, n=50, k=54, trans_a=False, trans_b=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["request", "request", "din", "serve", "pool", "pool", "fc", "fc", "bmm"])
    if kind in ("request", "serve"):
        c = dict(kind=kind, dtype=rng.choice(["f16", "f16", "f32"]), batch=_log(rng, 1 if kind == "request" else 64, 3000),
                 slots=rng.randint(4, 32), rows=_log(rng, 20_000, 1_000_000), dim=rng.choice([8, 12, 16, 18, 24, 32, 48, 64]),
                 mean_len=round(rng.uniform(1.0, 10.0), 2), zipf=round(rng.uniform(1.0, 1.2), 3), keyed=False,
                 dense=rng.randint(8, 64), h1=rng.choice([64, 100, 128, 200, 256, 400, 512]), h2=rng.choice([32, 40, 80, 100, 128, 256]))
        if rng.random() < 0.3:
            c.update(keyed=True, rows=_log(rng, 20_000, 100_000))
        if kind == "serve":
            c.update(predictors=16, passes=64)
        return c
    if kind == "din":
        return dict(kind=kind, dtype=rng.choice(["f16", "f16", "f32"]), batch=_log(rng, 1, 2000), hist=rng.randint(8, 60),
                    rows=_log(rng, 20_000, 2_000_000), dim=rng.choice([8, 12, 16, 18]), zipf=round(rng.uniform(1.0, 1.25), 3))
    if kind == "pool":
        dtype = rng.choice(["f32", "f16", "f16", "i8"])
        udf = rng.choice(["sum", "sum", "avg", "assign"])
        slots, dim = _log(rng, 1, 120), rng.choice([8, 16, 18, 24, 32, 48, 64, 100, 128, 200])
        trunc = rng.randint(5, 60) if udf == "assign" else 0
        mean_len = round(trunc * rng.uniform(0.3, 0.9) if trunc else rng.uniform(1.0, 24.0), 2)
        most = 6e8 / (slots * dim * (SIZE[dtype] * mean_len + 4 * max(trunc, 1)))  # samples whose rows and outputs are about 0.6 GB
        keyed = rng.random() < 0.3
        return dict(kind=kind, dtype=dtype, out=rng.choice(["f32", "f16"]), batch=_log(rng, 1, max(2, min(16384, int(most)))),
                    slots=slots, tables=min(slots, 4) if keyed else slots, rows=_log(rng, 20_000, 250_000 if keyed else 1_000_000),
                    dim=dim, mean_len=mean_len, zipf=rng.choice([0.0, 1.05, 1.1, 1.2]), keyed=keyed, udf=udf, trunc=trunc)
    if kind == "fc":
        dtype = rng.choice(["f16", "bf16", "f32"])
        k = _log(rng, 64, 4096)
        h1 = rng.choice([64, 80, 128, 200, 256, 400, 512, 768, 1024])
        most = (2e11 if dtype != "f32" else 2e10) / (2.0 * k * h1)
        return dict(kind=kind, dtype=dtype, batch=_log(rng, 1, min(16384, int(most))), k=k, h1=h1, h2=rng.choice([40, 80, 128, 256, 512]),
                    h3=rng.choice([0, 0, 32, 64, 200, 256]), n=rng.choice([1, 1, 2]), act=rng.choice(["relu", "prelu", "dice"]))
    if rng.random() < 0.3:  # a weighted sum over a history: one row times [history, channels]
        m, n, k = 1, rng.randint(8, 128), rng.randint(8, 200)
    else:
        m, n, k = _log(rng, 4, 200), _log(rng, 4, 200), _log(rng, 8, 128)
    return dict(kind=kind, dtype=rng.choice(["f16", "f16", "f32"]), batch=_log(rng, 1, min(4096, max(2, int(2e7 / (m * n + k * (m + n)))))), m=m,
                n=n, k=k, trans_a=rng.random() < 0.25, trans_b=rng.random() < 0.5)


# ---------------------------------------------------------------------------------------------- inputs
_CDF = {}


def _cdf(rows, zipf):
    """cumulative Zipf(zipf) over 1..rows; the last few are kept, many inputs being drawn from the same one"""
    if (rows, zipf) not in _CDF:
        while len(_CDF) > 3:
            _CDF.pop(next(iter(_CDF)))
        w = np.arange(1, rows + 1, dtype=np.float64)**(-zipf)
        _CDF[rows, zipf] = np.cumsum(w / w.sum())
    return _CDF[rows, zipf]


def _host_ids(rng, n, rows, zipf):
    rank = np.minimum(np.searchsorted(_cdf(rows, zipf), rng.random(n)), rows - 1).astype(np.int64)
    return (rank * 2654435761 + 12345) % rows  # hot rows scattered over the table


def _device_ids(gen, n, rows, zipf):
    if zipf == 0.0:
        return torch.randint(rows, (n, ), generator=gen, device="cuda")
    cdf = torch.from_numpy(_cdf(rows, zipf)).cuda()
    rank = torch.searchsorted(cdf, torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)).clamp_(max=rows - 1)
    return (rank * 2654435761 + 12345) % rows


def _distinct(rows, zipf, n):
    """expected number of distinct rows among n ids"""
    p = np.diff(_cdf(rows, zipf), prepend=0.0)
    return float(-np.expm1(n * np.log1p(-np.minimum(p, 0.999999))).sum())


def _keys(rng, n):
    """n distinct 62-bit keys"""
    return (np.arange(n, dtype=np.int64) << 40) | rng.integers(0, 1 << 40, n, dtype=np.int64)


def _table(gen, rows, dim, dtype, std=0.05):
    if dtype == "i8":
        return torch.randint(-127, 128, (rows, dim), generator=gen, device="cuda", dtype=torch.int8)
    return torch.empty((rows, dim), dtype=TORCH[dtype], device="cuda").normal_(0.0, std, generator=gen)


class _Ctr:
    """what ctr_model.build_manager reads of a configuration"""

    def __init__(self, case):
        self.dim, self.dense = case["dim"], case["dense"]
        self.in_dim = case["dense"] + case["slots"] * case["dim"]
        self.layers = (self.in_dim, case["h1"], case["h2"], 2)


def _ctr_manager(case, gen, rng):
    cfg = _Ctr(case)
    tables = [_table(gen, case["rows"], case["dim"], case["dtype"]) for _ in range(case["slots"])]
    mlp = []
    for k, n in zip(cfg.layers, cfg.layers[1:]):
        mlp.append((torch.from_numpy(rng.standard_normal((k, n), np.float32) / np.float32(math.sqrt(k))),
                    torch.from_numpy(rng.standard_normal(n, np.float32) * np.float32(0.1)), torch.full((n, ), 0.25)))
    dtype = np.float16 if case["dtype"] == "f16" else np.float32
    if not case["keyed"]:
        pm, fgs = ctr_model.build_manager(cfg, tables, mlp, dtype)
        return pm, fgs, None
    keys = [_keys(rng, case["rows"]) for _ in tables]
    # build_manager registers the tables by name: the keyed ones take the same names first, and a manager keeps the last
    pm, fgs = ctr_model.build_manager(cfg, tables, mlp, dtype)
    for (_, name, _), t, k in zip(fgs, tables, keys):
        pm.add_table(name, t, keys=k)
    return pm, fgs, keys


def _ctr_request(case, fgs, keys, rng):
    items = []
    for s, (fg, _, _) in enumerate(fgs):
        seg = np.clip(rng.poisson(case["mean_len"], case["batch"]), 1, 64).astype(np.int32)
        ids = _host_ids(rng, int(seg.sum()), case["rows"], case["zipf"])
        if keys is not None:
            known = rng.random(ids.size) >= 0.05  # some keys are in no table
            ids = np.where(known, keys[s][ids], -1 - ids)
        items += [(fg + ".ids", ids), (fg + ".values", np.ones(ids.size, np.float32)), (fg + ".segments", seg)]
    dense = rng.standard_normal((case["batch"], case["dense"]), np.float32)
    items.append(("dense", dense.astype(np.float16 if case["dtype"] == "f16" else np.float32)))
    return items


def _predictor(pm, items):
    """a predictor that has served the request's shapes once, and the request's argument arrays"""
    p = pm.create_predictor(1, 0)
    for name, a in items:
        p.feed(name, a)
    return p, p.feed_batch(items)


def _din_config(case):
    return din_model.Config3(batch=case["batch"], rows=case["rows"], T=case["hist"])


def prepare(case, seed):
    torch.cuda.set_device(0)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    return _PREPARE[case["kind"]](case, gen, rng)


def _prepare_request(case, gen, rng):
    pm, fgs, keys = _ctr_manager(case, gen, rng)
    p, batch = _predictor(pm, _ctr_request(case, fgs, keys, rng))
    return dict(run=_run_request, p=p, batch=batch)


def _prepare_din(case, gen, rng):
    cfg = _din_config(case)
    cfg.dim = case["dim"]
    d3, B, T = 3 * cfg.dim, case["batch"], case["hist"]
    weights = {}
    for tag, layers in (("att", (4 * d3, 80, 40, 1)), ("main", (3 * d3, 200, 80, 2))):
        weights[tag] = [dict(w=rng.standard_normal((k, n), np.float32) / np.float32(math.sqrt(k)),
                             b=rng.standard_normal(n, np.float32) * np.float32(0.1),
                             gamma=rng.standard_normal(n, np.float32) * np.float32(0.1),
                             mean=rng.standard_normal(n, np.float32) * np.float32(0.1),
                             var=rng.uniform(0.5, 1.5, n).astype(np.float32)) for k, n in zip(layers, layers[1:])]
    dtype = np.float16 if case["dtype"] == "f16" else np.float32
    tables = [_table(gen, case["rows"], cfg.dim, case["dtype"], 0.1) for _ in din_model.KINDS]
    pm, inputs = din_model.build_manager(cfg, tables, weights, dtype)
    seg = rng.integers(1, T + 1, B).astype(np.int32)
    feed = {"mask": (np.arange(T)[None, :] < seg[:, None]).astype(dtype).reshape(B, T, 1)}
    for kind in din_model.KINDS:
        for fg, s in ((kind, np.ones(B, np.int32)), (kind + "_his", seg.copy())):
            n = int(s.sum())
            feed[fg + ".ids"] = _host_ids(rng, n, case["rows"], case["zipf"])
            feed[fg + ".values"] = np.ones(n, np.float32)
            feed[fg + ".segments"] = s
    p, batch = _predictor(pm, [(name, feed[name]) for name in inputs])
    return dict(run=_run_request, p=p, batch=batch)


class _DeviceView:
    """a predictor's output blob as torch sees it"""

    def __init__(self, ptr, shape, dtype):
        self.__cuda_array_interface__ = dict(shape=shape, typestr=np.dtype(dtype).str, data=(ptr, False), version=3, strides=None)


def _prepare_serve(case, gen, rng):
    pm, fgs, keys = _ctr_manager(case, gen, rng)
    ps = [_predictor(pm, _ctr_request(case, fgs, keys, rng))[0] for _ in range(case["predictors"])]
    pool = pb.ServePool(SERVING_THREADS, 1)
    pool.run(ps, 2 * len(ps))
    outs = []
    for p in ps:
        outs.append(torch.as_tensor(_DeviceView(p.output_device_ptr("prob"), p.output_shape("prob"), p.output_dtype("prob")), device="cuda"))
        outs[-1].owner = p  # the memory is the predictor's: it lives as long as the view does
    return dict(run=_run_serve, pool=pool, ps=ps, passes=case["passes"], outs=outs)


def _prepare_pool(case, gen, rng):
    B, S = case["batch"], case["slots"]
    tables, keys = [], []
    for _ in range(case["tables"]):
        rows = _table(gen, case["rows"], case["dim"], case["dtype"])
        scale = None
        if case["dtype"] == "i8":
            scale = torch.empty(case["rows"], device="cuda").uniform_(1e-3, 1e-2, generator=gen)
        k = _keys(rng, case["rows"]) if case["keyed"] else None
        keys.append(torch.from_numpy(k).cuda() if k is not None else None)
        tables.append(bz.DeviceTable(rows, scale=scale, keys=k))
    seg = torch.poisson(torch.full((S, B), float(case["mean_len"]), device="cuda"), generator=gen).to(torch.int32)
    nnz = seg.sum(1).tolist()
    cols = case["dim"] * max(case["trunc"], 1)
    out = torch.zeros((B, S * cols), dtype=TORCH[case["out"]], device="cuda")
    items = []
    for s in range(S):
        ids = _device_ids(gen, max(nnz[s], 1), case["rows"], case["zipf"])
        key = keys[s % len(keys)]
        if key is not None:
            known = torch.rand(ids.numel(), generator=gen, device="cuda") >= 0.05
            ids = torch.where(known, key[ids], -1 - ids)
        items.append(dict(table=tables[s % len(tables)], ids=ids, values=torch.ones(ids.numel(), device="cuda"), segments=seg[s], nnz=nnz[s],
                          out=out, col=s * cols, udf=UDF[case["udf"]], trunc_dir=bz.ORDER, trunc_num=case["trunc"]))
    return dict(run=_run_pool, plan=bz.EmbeddingPlan(items), out=out)


def _prepare_fc(case, gen, rng):
    dt, tdt = {"f32": bz.F32, "f16": bz.F16, "bf16": bz.BF16}[case["dtype"]], TORCH[case["dtype"]]
    widths = [case["k"]] + [h for h in (case["h1"], case["h2"], case["h3"]) if h] + [case["n"]]
    x = torch.empty((case["batch"], case["k"]), device="cuda").normal_(generator=gen).to(tdt)
    layers, ys = [], []
    for k, n in zip(widths, widths[1:]):
        w = torch.empty((k, n), device="cuda").normal_(0.0, 1.0 / math.sqrt(k), generator=gen)
        params = {}
        if case["act"] == "prelu":
            params = dict(act=bz.ACT_PRELU, act_params=(torch.full((n, ), 0.25, device="cuda"), ))
        elif case["act"] == "dice":
            params = dict(act=bz.ACT_DICE, act_params=(torch.empty(n, device="cuda").normal_(0.0, 0.1, generator=gen),
                                                       torch.empty(n, device="cuda").normal_(0.0, 0.1, generator=gen),
                                                       torch.empty(n, device="cuda").uniform_(0.5, 1.5, generator=gen)))
        else:
            params = dict(act=bz.ACT_LEAKY_RELU, act_alpha=0.0)
        layers.append((bz.pack_weight(w, False, dt), k, torch.empty(n, device="cuda").normal_(0.0, 0.1, generator=gen), params))
        ys.append(torch.zeros((case["batch"], n), dtype=tdt, device="cuda"))
    prob = torch.zeros((case["batch"], case["n"]), dtype=torch.float32, device="cuda")
    return dict(run=_run_fc, x=x, layers=layers, ys=ys, prob=prob, act=bz.ACT_SOFTMAX if case["n"] > 1 else bz.ACT_SIGMOID)


def _prepare_bmm(case, gen, rng):
    dt = TORCH[case["dtype"]]
    B, m, n, k = (case[x] for x in ("batch", "m", "n", "k"))
    a = torch.empty((B, m * k), device="cuda").normal_(generator=gen).to(dt)
    b = torch.empty((B, n * k), device="cuda").normal_(generator=gen).to(dt)
    return dict(run=_run_bmm, a=a, b=b, c=torch.zeros((B, m, n), dtype=dt, device="cuda"), m=m, n=n, k=k, batch=B,
                ta=case["trans_a"], tb=case["trans_b"], alpha=1.0 / math.sqrt(k))


_PREPARE = dict(request=_prepare_request, din=_prepare_din, serve=_prepare_serve, pool=_prepare_pool, fc=_prepare_fc, bmm=_prepare_bmm)


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    return state["run"](state)


def _run_request(st):
    st["p"].feed_many(st["batch"])
    st["p"].forward()
    return st["p"].output_asnumpy("prob")


def _run_serve(st):
    st["pool"].run(st["ps"], st["passes"])
    return st["outs"]


def _run_pool(st):
    st["plan"].run()
    return st["out"]


def _run_fc(st):
    x, ys, layers = st["x"], st["ys"], st["layers"]
    last = len(layers) - 1
    in_head = layers[last - 1][0].shape[0] <= 256  # the layer before the head carries it in its launch, as a net runs a tower
    for i, (w, k, bias, params) in enumerate(layers[:last - 1 if in_head else last]):
        x = bz.fc_fused(x, w, k, bias=bias, out=ys[i], **params)
    w, k, bias, params = layers[last]
    if in_head:
        w1, k1, bias1, params1 = layers[last - 1]
        bz.fc_fused(x, w1, k1, bias=bias1, out=ys[last - 1], store_out=False, head=dict(w=w, bias=bias, act=st["act"], out=st["prob"]),
                    **params1)
        return ys[:last - 1], st["prob"]
    bz.fc_fused(x, w, k, bias=bias, out=st["prob"], act=st["act"])
    return ys[:last], st["prob"]


def _run_bmm(st):
    return bz.gemm_strided_batched(st["a"], st["b"], st["c"], st["m"], st["n"], st["k"], st["batch"], st["m"] * st["k"],
                                   st["n"] * st["k"], st["m"] * st["n"], trans_a=st["ta"], trans_b=st["tb"], alpha=st["alpha"])


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _lookup_bytes(nnz, batch, rows, zipf, row_bytes):
    """one slot: ids, values and counts once, each distinct row once"""
    return 12.0 * nnz + 4.0 * batch + row_bytes * _distinct(rows, zipf, nnz)


def _tower(batch, widths, es):
    """(bytes of the weights, flops) of a stack of FC layers"""
    pairs = list(zip(widths, widths[1:]))
    return float(sum(k * n * es for k, n in pairs)), float(sum(2 * batch * k * n for k, n in pairs))


def work(case):
    kind, B = case["kind"], case["batch"]
    es = SIZE[case["dtype"]]
    if kind in ("request", "serve"):
        wb, fl = _tower(B, _Ctr(case).layers, es)
        by = case["slots"] * _lookup_bytes(case["mean_len"] * B, B, case["rows"], case["zipf"], case["dim"] * es)
        by += B * (case["dense"] + 2) * es
        n = case["passes"] if kind == "serve" else 1
        return {"bytes": n * by + wb, "flops": n * fl}
    if kind == "din":
        T, d3 = case["hist"], 3 * case["dim"]
        w1, f1 = _tower(B * T, (4 * d3, 80, 40, 1), es)
        w2, f2 = _tower(B, (3 * d3, 200, 80, 2), es)
        nnz = B * (T + 1) / 2
        by = 3 * (_lookup_bytes(nnz, B, case["rows"], case["zipf"], case["dim"] * es) + 16.0 * B) + B * (T + 2) * es
        return {"bytes": by + w1 + w2, "flops": f1 + f2 + 4.0 * B * T * d3}
    if kind == "pool":
        nnz = case["mean_len"] * B
        per_table = case["slots"] / case["tables"]
        by = case["slots"] * (12.0 * nnz + 4.0 * B)
        by += case["tables"] * _distinct(case["rows"], case["zipf"], nnz * per_table) * (case["dim"] * es + (4 if case["dtype"] == "i8" else 0))
        by += B * case["slots"] * case["dim"] * max(case["trunc"], 1) * SIZE[case["out"]]
        return {"bytes": by, "flops": 2.0 * nnz * case["slots"] * case["dim"]}
    if kind == "fc":
        widths = [case["k"]] + [h for h in (case["h1"], case["h2"], case["h3"]) if h] + [case["n"]]
        wb, fl = _tower(B, widths, es)
        return {"bytes": wb + B * (case["k"] + sum(widths[1:-2] if widths[-2] <= 256 else widths[1:-1])) * es + B * case["n"] * 4.0, "flops": fl}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": float(B * (m * k + n * k + m * n) * es), "flops": 2.0 * B * m * n * k}


def tolerance(case):
    """what the data types give: 2-byte tensors are rounded between operators, fp32 ones differ by the order of their sums"""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "pool":  # sums are added in the ids' order whatever the kernel: no more than the rounding of the output
        return {"rel": {"f32": 1e-6, "f16": 5e-4, "bf16": 4e-3}[case["out"]]}
    return {"rel": {"f32": 1e-5, "f16": 3e-3, "bf16": 1e-2}[dtype]}
