"""GPU tests of the drop-in boundary: operators run through Predictor / the Blaze_* C ABI.

The reference's operator tests build a net from a text NetDef whose inputs are ConstantFill ops, run it and compare
outputs with |d| <= 1e-6 (test/operator/operator_test_common.h:20-84).  The same is done here from the same data
(tests/golden/reference_kats.json), through Blaze_PredictorManagerLoadModelFromString / Blaze_PredictorCreate /
Blaze_PredictorForward / Blaze_PredictorOutput on device_type 1.
"""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def pb():
    import torch
    import blaze_hip
    import pyblaze_hip
    assert torch.cuda.is_available(), "no GPU visible"
    blaze_hip.device_check()
    return pyblaze_hip


def _np_dtype(code):
    return {1: np.float32, 2: np.int32, 10: np.int64, 12: np.float16}[code]


def _net_from_kat(pb, case, skip_types=()):
    nb = pb.NetBuilder("kat", device_type=1)
    for name, t in case["tensors"].items():
        nb.constant(name, np.array(t["values"], _np_dtype(t["dtype"])).reshape(t["shape"]), dtype=t["dtype"])
    for op in case["ops"]:
        args = {}
        for k, v in op["args"].items():
            if k in ("store_name", "store_type", "store_url"):
                continue
            if k in ("alpha", "beta"):
                v = float(v)
            args[k] = v
        nb.op(op["type"], op["inputs"], op["outputs"], **args)
    for name, e in case["expected"].items():
        nb.external_output(name, e["dtype"])
    return nb.text()


DENSE = ["gemm_net_v1_cpu", "prelu_net_v1_cpu", "dice_net_v1_cpu", "leaky_relu_net_v1_cpu", "sigmoid_net_v1_cpu",
         "softmax_net_v1_cpu", "matmul_net_v1_cpu", "fused_parallel_gemm_net_v1_cpu", "fused_parallel_gemm_net_v2_cpu",
         "fused_parallel_gemm_net_v3_cpu", "fused_parallel_gemm_net_v4_cpu", "fused_parallel_gemm_net_v5_cpu",
         "fused_parallel_matmul_net_v1_cpu", "fused_parallel_matmul_net_v2_cpu", "fused_parallel_matmul_net_v3_cpu",
         "concat_net_v1_cpu", "concat_net_v2_cpu", "reduce_sum_net_v1_cpu", "fuse_net_v1_cpu", "fuse_net_v2_cpu",
         "reshape_net_v1_cpu", "batch_normalization_net_v1_cpu", "elementwise_add_net_v1_cpu", "elementwise_add_net_v2_cpu",
         "elementwise_sub_net_v1_cpu", "elementwise_sub_net_v2_cpu", "elementwise_mul_net_v1_cpu", "elementwise_mul_net_v2_cpu",
         "elementwise_div_net_v1_cpu", "elementwise_div_net_v2_cpu", "elementwise_broadcast_to_net_v1_cpu",
         "elementwise_broadcast_to_net_v2_cpu", "elementwise_where_net_v1_cpu", "split_net_v1_cpu", "split_net_v2_cpu",
         "gather_net_v1_cpu", "gather_net_v2_cpu", "slice_net_v1_cpu"]


@pytest.mark.parametrize("name", DENSE)
def test_reference_operator_kats_through_predictor(pb, kats, name):
    case = kats[name]
    pm = pb.PredictorManager()
    pm.load_model_from_string(_net_from_kat(pb, case), True)
    p = pm.create_predictor(1, 0)
    print("case", name, flush=True)
    p.register_observers(["profile"])
    p.forward()
    for out_name, e in case["expected"].items():
        got = p.output_asnumpy(out_name)
        assert list(got.shape) == e["shape"]
        np.testing.assert_allclose(got, np.array(e["values"], np.float32).reshape(e["shape"]), rtol=0, atol=1e-6)
    if name.startswith("fused_parallel_gemm"):
        # the parallel_num sibling FCs go out as one launch (the reference: one GemmStridedBatched, fused_parallel_gemm_op.h:115-129)
        ev = [e for e in json.loads(p.dump_observers()["profile"])["traceEvents"] if e["name"].startswith("FusedParallelGemm")]
        assert len(ev) == 1 and ev[0]["args"]["launches"] == 1, ev


def test_reference_embedding_kat_through_predictor(pb, kats):
    """embedding_v1.conf: the reference runs it over its mock puller (every key -> a row of ones); here the device
    store gets tables of ones keyed by every id of the fixture."""
    case = kats["embedding_v1"]
    pm = pb.PredictorManager()
    for fg, table, dim in (("101", "a_01", 4), ("102", "a_02", 8), ("104_7", "a_03", 6)):
        ids = np.unique(np.array(case["tensors"][fg + ".ids"]["values"], np.int64))
        pm.add_table(table, np.ones((ids.size, dim), np.float32), keys=ids)
    pm.load_model_from_string(_net_from_kat(pb, case), True)
    p = pm.create_predictor(1, 0)
    p.forward()
    for out_name, e in case["expected"].items():
        got = p.output_asnumpy(out_name)
        assert list(got.shape) == e["shape"] and got.dtype == np.float32
        np.testing.assert_allclose(got, np.array(e["values"], np.float32).reshape(e["shape"]), rtol=0, atol=1e-6)


def _write_csv(path, keys, rows):
    with open(path, "w") as f:
        for k, r in zip(keys, rows):
            f.write(",".join([str(int(k))] + [repr(float(x)) for x in r]) + "\n")


def _ctr_text(pb, fgs, blocks, dims_in, layers, acts, dtype, fuse, dense_name="dense"):
    """Embedding -> Concat(dense, block) -> [Gemm + activation]* ; returns (text, weights)."""
    code = pb.K_FLOAT16 if dtype == np.float16 else pb.K_FLOAT
    nb = pb.NetBuilder("ctr", device_type=1)
    inputs = []
    for fg, _, _ in fgs:
        nb.external_input(fg + ".ids", pb.K_INT64)
        nb.external_input(fg + ".values", pb.K_FLOAT)
        nb.external_input(fg + ".segments", pb.K_INT32)
        inputs += [fg + ".ids", fg + ".values", fg + ".segments"]
    nb.external_input(dense_name, code)
    nb.external_output("prob", code)
    nb.arg("fuse_gemm_activation", int(fuse))
    rng = np.random.default_rng(77)
    weights = []
    for li in range(len(layers) - 1):
        k, n = layers[li], layers[li + 1]
        w = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)
        b = (rng.standard_normal(n) * 0.1).astype(np.float32)
        extra = ()
        if acts[li] == "PRelu":
            extra = (rng.uniform(0.1, 0.4, n).astype(np.float32), )
        elif acts[li] == "Dice":
            extra = ((rng.standard_normal(n) * 0.1).astype(np.float32), (rng.standard_normal(n) * 0.1).astype(np.float32),
                     rng.uniform(0.5, 1.5, n).astype(np.float32))
        weights.append((w, b, extra))
        nb.constant("w%d" % li, w, dtype=code)
        nb.constant("b%d" % li, b, dtype=code)
        for j, e in enumerate(extra):
            nb.constant("p%d_%d" % (li, j), e, dtype=code)
    nb.op("Embedding", inputs, ["block"], embedding_config=pb.embedding_config_text(fgs, blocks),
          **({"out_dtype": code} if dtype == np.float16 else {}))
    nb.op("Concat", [dense_name, "block"], ["x0"], axis=1)
    for li in range(len(layers) - 1):
        last = li == len(layers) - 2
        nb.op("Gemm", ["x%d" % li, "w%d" % li, "b%d" % li], ["h%d" % li])
        out = "prob" if last else "x%d" % (li + 1)
        if acts[li] == "Softmax":
            nb.op("Softmax", ["h%d" % li], [out], axis=1)
        elif acts[li] == "LeakyRelu":
            nb.op("LeakyRelu", ["h%d" % li], [out], alpha=0.0)
        elif acts[li] == "Sigmoid":
            nb.op("Sigmoid", ["h%d" % li], [out])
        else:
            nb.op(acts[li], ["h%d" % li] + ["p%d_%d" % (li, j) for j in range(len(weights[li][2]))], [out])
    return nb.text(), weights


def _oracle_ctr(oracle, tables, fgs, blocks, inputs, dense, weights, acts, r):
    """The same net on the CPU oracle; r rounds to the model's storage type after every op (identity for fp32)."""
    outs = oracle.embedding_op({fg: (t, d) for fg, t, d in fgs}, blocks, inputs, tables)
    h = np.concatenate([r(dense), r(outs[0])], axis=1)
    for (w, b, extra), act in zip(weights, acts):
        y = r(oracle.gemm_op(h, r(w), r(b)))
        if act == "PRelu":
            y = oracle.prelu(y, r(extra[0]))
        elif act == "Dice":
            y = oracle.dice(y, *[r(e) for e in extra])
        elif act == "LeakyRelu":
            y = oracle.leaky_relu(y, 0.0)
        elif act == "Sigmoid":
            y = oracle.sigmoid(y)
        else:
            y = oracle.softmax(y, 1)
        h = r(y)
    return h


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("acts", [("PRelu", "Dice", "Softmax"), ("LeakyRelu", "Sigmoid", "Softmax")])
def test_ctr_model_from_qed_file_fused_and_unfused(pb, oracle, tmp_path, dtype, acts):
    """Text tables -> Blaze_QuickEmbeddingBuild* -> Blaze_LoadSparseModelWeight -> Embedding + Concat + FC stack.
    With and without folding the activations into the Gemm epilogue; both against the oracle."""
    rng = np.random.default_rng(5)
    fgs = [("101", "t_a", 8), ("102", "t_b", 16), ("103", "t_c", 8)]
    blocks = [[dict(fg="101", udf=0), dict(fg="102", udf=1), dict(fg="103", udf=0)]]
    tabs, oracle_tabs = {}, {}
    for _, tname, dim in fgs:
        n = int(rng.integers(30, 120))
        keys = np.unique(rng.integers(-2**40, 2**40, n * 2, dtype=np.int64))[:n]
        rows = (rng.standard_normal((n, dim)) * 0.5).astype(np.float32)
        _write_csv(tmp_path / tname, keys, rows)
        tabs[tname] = (keys, rows)
    open(tmp_path / "meta", "w").write("".join(t + "\n" for _, t, _ in fgs))
    qed = str(tmp_path / "model.qed")
    pb.build_qed(str(tmp_path), "meta", qed, fp16=(dtype == np.float16))
    for tname, (keys, rows) in tabs.items():
        # what the builder parsed back from text (repr round-trips fp32 exactly), narrowed for the fp16 file
        oracle_tabs[tname] = oracle.Table(rows.astype(np.float16) if dtype == np.float16 else rows, keys=keys)
    batch, dense_dim = 37, 5
    layers = (dense_dim + 32, 24, 16, 2)
    inputs = {}
    for fg, tname, _ in fgs:
        seg = rng.integers(0, 6, batch).astype(np.int32)
        pool = np.concatenate([tabs[tname][0], rng.integers(-2**40, 2**40, 10, dtype=np.int64)])
        ids = rng.choice(pool, int(seg.sum()))
        inputs[fg] = (ids.astype(np.int64), rng.standard_normal(ids.size).astype(np.float32), seg)
    dense = rng.standard_normal((batch, dense_dim)).astype(np.float32)
    r = (lambda x: np.asarray(x, np.float32).astype(np.float16).astype(np.float32)) if dtype == np.float16 else (lambda x: x)
    results = []
    for fuse in (True, False):
        text, weights = _ctr_text(pb, fgs, blocks, dense_dim, layers, acts, dtype, fuse)
        pm = pb.PredictorManager()
        pm.load_sparse_model_weight(qed)
        pm.load_model_from_string(text, True)
        p = pm.create_predictor(1, 0)
        assert p.list_input_names() == [n for fg, _, _ in fgs for n in (fg + ".ids", fg + ".values", fg + ".segments")] + ["dense"]
        assert p.list_output_names() == ["prob"]
        for fg, (ids, vals, seg) in inputs.items():
            p.feed(fg + ".ids", ids)
            p.feed(fg + ".values", vals)
            p.feed(fg + ".segments", seg)
        p.feed("dense", dense.astype(dtype))
        print("case dtype=%s acts=%s fuse=%s" % (dtype.__name__, acts, fuse), flush=True)
        p.forward()
        got = p.output_asnumpy("prob")
        assert got.shape == (batch, 2) and got.dtype == dtype
        results.append(got.astype(np.float32))
        p.forward()  # a second run reuses cached descriptors and packed weights
        assert np.array_equal(p.output_asnumpy("prob").astype(np.float32), results[-1])
    want = _oracle_ctr(oracle, oracle_tabs, fgs, blocks, inputs, dense, weights, acts, r)
    tol = 2e-3 if dtype == np.float16 else 1e-5
    for got in results:
        np.testing.assert_allclose(got, want, rtol=tol, atol=tol)
    np.testing.assert_allclose(results[0], results[1], rtol=tol, atol=tol)
    names = p.list_internal_names()
    assert "w0" in names and p.internal_shape("w0") == (layers[0], layers[1])
    np.testing.assert_array_equal(p.internal_asnumpy("w0"), weights[0][0].astype(dtype))


def test_feed_and_forward_error_conventions(pb):
    pm = pb.PredictorManager()
    nb = pb.NetBuilder("err", device_type=1)
    nb.external_input("x", pb.K_FLOAT)
    nb.external_output("y")
    nb.constant("w", np.ones((4, 3), np.float32))
    nb.op("Gemm", ["x", "w"], ["y"])
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    x = np.ones((2, 4), np.float32)
    p.reshape_input("x", x.shape)
    with pytest.raises(pb.BlazeError, match="Feed x failed"):
        p.feed_raw("x", x, x.nbytes - 4)  # len must equal size * sizeof(dtype)
    with pytest.raises(pb.BlazeError, match="Feed nope failed"):
        p.feed_raw("nope", x, x.nbytes)
    p.feed("x", x)
    p.forward()
    np.testing.assert_array_equal(p.output_asnumpy("y"), np.full((2, 3), 4, np.float32))
    p.feed("x", np.ones((2, 5), np.float32))  # inner dimension no longer matches the weight
    with pytest.raises(pb.BlazeError, match="Forward failed.*a_k=5 b_k=4"):
        p.forward()
    p.feed("x", x)  # the predictor stays usable after a failed run
    p.forward()
    np.testing.assert_array_equal(p.output_asnumpy("y"), np.full((2, 3), 4, np.float32))
    p.register_observers(["profile"])
    p.forward()
    trace = json.loads(p.dump_observers()["profile"])
    assert [e["name"].split(":")[0] for e in trace["traceEvents"]] == ["ConstantFill", "Gemm"]


def test_embedding_operator_errors(pb):
    cfg = pb.embedding_config_text([("101", "t", 4)], [[dict(fg="101", udf=0)]])

    def build(cfg_text, store=True, inputs=("101.ids", "101.values", "101.segments")):
        pm = pb.PredictorManager()
        if store:
            pm.add_table("t", np.ones((3, 4), np.float32))
        nb = pb.NetBuilder("e", device_type=1)
        for n, dt in zip(inputs, (pb.K_INT64, pb.K_FLOAT, pb.K_INT32)):
            nb.external_input(n, dt)
        nb.external_output("block")
        nb.op("Embedding", list(inputs), ["block"], embedding_config=cfg_text)
        pm.load_model_from_string(nb.text(), True)
        return pm

    with pytest.raises(pb.BlazeError, match="Parse embedding config failed"):
        build("feature_group_config { feature_group : ").create_predictor(1, 0)
    with pytest.raises(pb.BlazeError, match="feature group config not exist"):
        build(pb.embedding_config_text([("101", "t", 4)], [[dict(fg="999", udf=0)]])).create_predictor(1, 0)
    with pytest.raises(pb.BlazeError, match="id input name"):
        build(cfg, inputs=("101.ids", "102.values", "101.segments")).create_predictor(1, 0)
    p = build(cfg, store=False).create_predictor(1, 0)
    p.feed("101.ids", np.array([0, 1], np.int64))
    p.feed("101.values", np.ones(2, np.float32))
    p.feed("101.segments", np.array([2], np.int32))
    with pytest.raises(pb.BlazeError, match="no sparse puller"):
        p.forward()
    p = build(cfg).create_predictor(1, 0)
    p.feed("101.ids", np.array([0, 1], np.int64))
    p.feed("101.values", np.ones(3, np.float32))  # ids / values disagree
    p.feed("101.segments", np.array([2], np.int32))
    with pytest.raises(pb.BlazeError, match="id_blob->size"):
        p.forward()
    p.feed("101.values", np.array([2.0, 3.0], np.float32))
    p.forward()
    np.testing.assert_array_equal(p.output_asnumpy("block"), np.full((1, 4), 5.0, np.float32))
    # unknown table name: the block stays zero
    p = build(pb.embedding_config_text([("101", "unknown_table", 4)], [[dict(fg="101", udf=0)]])).create_predictor(1, 0)
    p.feed("101.ids", np.array([0, 1], np.int64))
    p.feed("101.values", np.ones(2, np.float32))
    p.feed("101.segments", np.array([2], np.int32))
    p.forward()
    assert not p.output_asnumpy("block").any()


def test_concat_inputs_written_in_place_give_identical_results(pb):
    """Concat(dense, block) whose inputs are an external input and an Embedding block read by nothing else: both
    live inside the Concat's output (the Feed copies rows at that tensor's pitch, the pooling kernel writes at it)
    and nothing is copied.  Bit-identical to the net with the aliasing switched off, also after the batch size and
    the fed data change."""
    import torch
    from ctr_model import build_manager, feed_inputs
    from synth import Config2
    cfg = Config2(batch=257, rows=3000, slots=26)
    tables, mlp = cfg.tables(), cfg.mlp()
    sparse, dense = cfg.batches(2)
    small = Config2(batch=64, rows=3000, slots=26)
    sparse_s, dense_s = small.batches(1, seed_offset=9)
    outs = {}
    for alias in (1, 0):
        pm, fgs = build_manager(cfg, tables, mlp, np.float16, net_args={"alias_concat_inputs": alias})
        p = pm.create_predictor(1, 0)
        got = []
        for sp, dn in ((sparse[0], dense[0]), (sparse_s[0], dense_s[0]), (sparse[1], dense[1])):  # batch 257 -> 64 -> 257
            feed_inputs(p, fgs, sp, dn, np.float16)
            p.forward()
            got.append(p.output_asnumpy("prob").copy())
        outs[alias] = got
        if alias:
            with pytest.raises(pb.BlazeError):
                p.input_device_ptr("dense")  # a strided input has no plain buffer to hand out
        else:
            assert p.input_device_ptr("dense")
    torch.cuda.synchronize()
    for a, b in zip(outs[1], outs[0]):
        assert a.shape == b.shape and np.array_equal(a.view(np.uint16), b.view(np.uint16))
    assert outs[1][0].shape == (257, 2) and outs[1][1].shape == (64, 2)


def test_forward_in_two_halves_and_serve_pool_match_plain_forward(pb):
    """ForwardLaunch / ForwardWait keep two predictors of one thread queued at once, and the serving pool does the
    same inside the library (depth 2) or calls plain Forward (depth 1): every predictor ends with bit-identical
    probabilities to its own synchronous Forward.  ForwardWait without a launch is an error, not a hang."""
    import torch
    from ctr_model import build_manager, make_predictor
    from synth import Config2
    cfg = Config2(batch=200, rows=3000, slots=26)
    tables, mlp = cfg.tables(), cfg.mlp()
    sparse, dense = cfg.batches(4)
    pm, fgs = build_manager(cfg, tables, mlp, np.float16)
    preds = [make_predictor(pm, fgs, sparse[b], dense[b], np.float16) for b in range(4)]
    want = []
    for p in preds:
        p.forward()
        want.append(p.output_asnumpy("prob").copy())
    assert not np.array_equal(want[0], want[1])  # different batches: a mixed-up predictor would show

    with pytest.raises(pb.BlazeError, match="ForwardWait without a ForwardLaunch"):
        preds[0].forward_wait()
    preds[0].forward_launch()
    preds[1].forward_launch()
    preds[0].forward_wait()
    preds[1].forward_wait()
    preds[2].forward_launch()
    preds[2].forward()  # a launch nobody waited for is waited for by the next Forward
    for b in range(3):
        np.testing.assert_array_equal(preds[b].output_asnumpy("prob"), want[b])

    for threads, depth, steps in ((2, 1, 13), (2, 2, 13), (1, 4, 9), (4, 2, 6), (2, 2, 1), (2, 2, 0)):
        print("serve pool threads=%d depth=%d steps=%d" % (threads, depth, steps), flush=True)
        pool = pb.ServePool(threads, depth)
        pool.run(preds, steps)
        torch.cuda.synchronize()
        for b in range(4):
            np.testing.assert_array_equal(preds[b].output_asnumpy("prob"), want[b])
        # one latency per pass of the job (launch to the return of its wait), positive and well under a second
        lat = pool.latencies_ms()
        assert lat.shape == (steps, ) and (steps == 0 or (lat.min() > 0 and lat.max() < 1000.0)), lat
        del pool
    with pytest.raises(pb.BlazeError, match="multiple of the pool's threads"):
        pb.ServePool(3).run(preds, 4)
    # the serving threads (and their streams) are gone; destroying predictors whose last passes ran on those streams
    # must not leave a runtime error behind for the caller's next GPU call
    import gc
    preds[0].forward_launch()  # one pass still in flight at destruction, on this thread's stream
    del preds, p
    gc.collect()
    assert float(torch.ones(4, device="cuda").sum()) == 4.0
    torch.cuda.synchronize()


def test_serve_pool_spreads_its_streams_evenly_over_the_hardware_queues(pb):
    """The pool creates its threads' streams and measures which of them share a hardware queue: every queue it saw
    serves as many threads as any other, give or take one, whatever streams the process holds besides (some idle ones
    are created first), and neighbouring threads sit on different queues.  Results are the plain Forward's."""
    import collections
    import torch
    from ctr_model import build_manager, make_predictor
    from synth import Config2
    cfg = Config2(batch=64, rows=500, slots=26)
    tables, mlp = cfg.tables(), cfg.mlp()
    sparse, dense = cfg.batches(8)
    pm, fgs = build_manager(cfg, tables, mlp, np.float16)
    preds = [make_predictor(pm, fgs, sparse[b], dense[b], np.float16) for b in range(8)]
    want = []
    for p in preds:
        p.forward()
        want.append(p.output_asnumpy("prob").copy())
    idle = [torch.cuda.Stream() for _ in range(3)]  # streams of the process that serve nothing
    for st in idle:
        with torch.cuda.stream(st):
            torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    for threads in (8, 4, 2, 1):
        pool = pb.ServePool(threads, 1)
        assert pool.stream_queues() == []
        pool.run(preds, 16)
        q = pool.stream_queues()
        print("threads", threads, "queues", q, flush=True)
        assert len(q) == threads
        per_queue = collections.Counter(q)
        assert max(per_queue.values()) - min(per_queue.values()) <= 1, q
        assert len(per_queue) >= min(threads, 2), q  # (the runtime's default is 4 queues)
        if threads > 1 and len(per_queue) > 1:
            assert all(q[t] != q[t + 1] for t in range(threads - 1)), q
        pool.run(preds, 8)
        assert pool.stream_queues() == q  # measured once
        for b in range(8):
            np.testing.assert_array_equal(preds[b].output_asnumpy("prob"), want[b])
        del pool


def test_skinny_last_layer_rides_in_the_launch_before_it(pb, oracle):
    """Gemm+PRelu (512 -> 256) followed by Gemm+Softmax (256 -> 2): by default the second runs inside the first one's
    launch (bz_fc_desc.head_*) and the 256-wide tensor between them is never stored; fuse_fc_head: 0 runs them one by
    one.  Same probabilities to 2e-3 (the fused tile sums in another order), also after the batch size changes."""
    import torch
    from ctr_model import build_manager, feed_inputs
    from synth import Config2
    cfg = Config2(batch=300, rows=4000, slots=26)
    small = Config2(batch=33, rows=4000, slots=26)
    tables, mlp = cfg.tables(), cfg.mlp()
    sparse, dense = cfg.batches(2)
    sparse_s, dense_s = small.batches(1, seed_offset=4)
    probs = {}
    for fuse in (1, 0):
        pm, fgs = build_manager(cfg, tables, mlp, np.float16, net_args={"fuse_fc_head": fuse})
        p = pm.create_predictor(1, 0)
        p.register_observers(["profile"])
        got = []
        for sp, dn in ((sparse[0], dense[0]), (sparse_s[0], dense_s[0]), (sparse[1], dense[1])):
            feed_inputs(p, fgs, sp, dn, np.float16)
            p.forward()
            got.append(p.output_asnumpy("prob").astype(np.float32))
        ran = [e["name"].split(":")[0] for e in json.loads(p.dump_observers()["profile"])["traceEvents"] if e["dur"] > 0]
        assert ran.count("Gemm") == (2 if fuse else 3), ran
        probs[fuse] = got
    torch.cuda.synchronize()
    for a, b, n in zip(probs[1], probs[0], (300, 33, 300)):
        assert a.shape == (n, 2)
        np.testing.assert_allclose(a, b, rtol=2e-3, atol=2e-3)
        np.testing.assert_allclose(a.sum(1), 1.0, rtol=2e-3)
    assert not np.array_equal(probs[1][0], probs[1][2])


def test_embedding_operator_scans_first_when_the_batch_is_large(pb):
    """A batch so large that every workgroup of the pooling kernel would re-read tens of thousands of counts: the
    puller follows the planner's advice, scans the segments in a launch of their own and pools from the offsets.
    Bit-identical block to the one-launch form of the kernel layer."""
    import torch
    import blaze_hip as bz
    from ctr_model import build_manager, make_predictor
    from synth import Config2
    cfg = Config2(batch=70000, rows=5000, slots=2)
    tables, mlp = cfg.tables(), cfg.mlp()
    sparse, dense = cfg.batches(1)
    pm, fgs = build_manager(cfg, tables, mlp, np.float16, expose_block=True)
    p = make_predictor(pm, fgs, sparse[0], dense[0], np.float16)
    p.forward()
    got = p.output_asnumpy("block")
    out = torch.zeros((cfg.batch, cfg.slots * cfg.dim), dtype=torch.float16, device="cuda")
    items, keep = [], []
    for s, (ids, vals, seg) in enumerate(sparse[0]):
        t = [torch.from_numpy(x).cuda() for x in (ids, vals, seg)]
        keep.append(t)
        items.append(dict(table=bz.DeviceTable(tables[s]), ids=t[0], values=t[1], segments=t[2], out=out, col=s * cfg.dim, udf=bz.SUM))
    auto = bz.EmbeddingPlan(items)
    assert auto.launch.fused_scan == 0  # the same advice the puller received
    bz.EmbeddingPlan(items, fused_scan=True).run()
    torch.cuda.synchronize()
    assert got.shape == (cfg.batch, cfg.slots * cfg.dim) and got.any()
    assert np.array_equal(got.view(np.uint16), out.cpu().numpy().view(np.uint16))
    assert p.output_asnumpy("prob").shape == (cfg.batch, 2)


def test_feed_many_equals_feeding_one_by_one(pb):
    """Blaze_PredictorFeedMany: all inputs in one call, the plain device inputs in one transfer through an arena the
    input tensors then view.  Same probabilities as feeding one by one -- after the first call, after the batch grows
    (the arena is outgrown), after it shrinks, and when single Feed calls follow on the re-viewed tensors; a wrong
    length is refused with the reference's message."""
    from ctr_model import build_manager, feed_inputs
    from synth import Config2

    def items_of(fgs, sp, dn):
        items = []
        for (fg, _, _), (ids, vals, seg) in zip(fgs, sp):
            items += [(fg + ".ids", ids), (fg + ".values", vals), (fg + ".segments", seg)]
        return items + [("dense", dn.astype(np.float16))]

    base = Config2(batch=64, rows=3000, slots=26)
    tables, mlp = base.tables(), base.mlp()
    pm, fgs = build_manager(base, tables, mlp, np.float16)
    one, many = pm.create_predictor(1, 0), pm.create_predictor(1, 0)
    for batch, seed in ((64, 0), (300, 3), (17, 5), (300, 7)):
        cfg = Config2(batch=batch, rows=3000, slots=26)
        sparse, dense = cfg.batches(1, seed_offset=seed)
        feed_inputs(one, fgs, sparse[0], dense[0], np.float16)
        one.forward()
        want = one.output_asnumpy("prob").copy()
        items = items_of(fgs, sparse[0], dense[0])
        for name, a in items:
            many.reshape_input(name, a.shape)
        fb = many.feed_batch(items)
        for _ in range(2):  # the second call finds the tensors already viewing the arena
            many.feed_many(fb)
            many.forward()
            np.testing.assert_array_equal(many.output_asnumpy("prob"), want)
    # single feeds on tensors that view the arena
    sparse, dense = Config2(batch=300, rows=3000, slots=26).batches(1, seed_offset=11)
    feed_inputs(one, fgs, sparse[0], dense[0], np.float16)
    one.forward()
    many.feed("fg00.values", sparse[0][0][1])          # same shape as before: reshape + Feed
    for name, a in items_of(fgs, sparse[0], dense[0]):
        many.feed(name, a)
    many.forward()
    np.testing.assert_array_equal(many.output_asnumpy("prob"), one.output_asnumpy("prob"))
    bad = many.feed_batch([("fg00.segments", np.zeros(7, np.int32))])
    with pytest.raises(pb.BlazeError, match="FeedMany failed"):
        many.feed_many(bad)


def test_threads_feeding_alternating_requests_get_their_own_results(pb):
    """Four serving threads, a predictor each, every step another request (two request sizes alternate, so the feed
    arena's layout, the tensors' addresses and the pooling kernel's slot records change every step) through
    FeedMany + Forward + Output: every result equals the one computed for that request alone."""
    import threading
    from ctr_model import build_manager, feed_inputs
    from synth import Config2
    base = Config2(batch=128, rows=3000, slots=26)
    tables, mlp = base.tables(), base.mlp()
    pm, fgs = build_manager(base, tables, mlp, np.float16)
    requests = []
    ref = pm.create_predictor(1, 0)
    for batch, seed in ((128, 1), (61, 2), (128, 3), (200, 4)):
        cfg = Config2(batch=batch, rows=3000, slots=26)
        sparse, dense = cfg.batches(1, seed_offset=seed)
        feed_inputs(ref, fgs, sparse[0], dense[0], np.float16)
        ref.forward()
        items = []
        for (fg, _, _), (ids, vals, seg) in zip(fgs, sparse[0]):
            items += [(fg + ".ids", ids), (fg + ".values", vals), (fg + ".segments", seg)]
        items.append(("dense", dense[0].astype(np.float16)))
        requests.append((items, ref.output_asnumpy("prob").copy()))
    errors = []

    def worker(t):
        try:
            p = pm.create_predictor(1, 0)
            batches = [p.feed_batch(items) for items, _ in requests]
            for i in range(60):
                r = (i + t) % len(requests)
                for name, a in requests[r][0]:
                    p.reshape_input(name, a.shape)
                p.feed_many(batches[r])
                p.forward()
                got = p.output_asnumpy("prob")
                if not np.array_equal(got, requests[r][1]):
                    errors.append("thread %d step %d request %d: max diff %g" % (t, i, r, np.abs(got.astype(np.float32) - requests[r][1].astype(np.float32)).max()))
                    return
        except Exception as e:  # noqa: BLE001
            errors.append("thread %d: %r" % (t, e))

    threads = [threading.Thread(target=worker, args=(t, )) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors


def test_optimized_model_file_gives_the_same_outputs(pb, oracle, tmp_path):
    """NetDef -> NetDef: Blaze_OptimizeBlaze rewrites three sibling Gemms (constant weights and biases of one shape)
    into FusedParallelGemm + Split; the optimized model file, loaded through Blaze_PredcitorManagerLoadModel, gives the
    outputs of the original one and of the oracle, with one FC launch and a Split that copies nothing.  Also the
    reference's own fixture (tests/golden/pattern/parallel_gemm_fusion.blaze, moved to the device)."""
    import json
    rng = np.random.default_rng(11)
    M, K, N, P = 37, 24, 16, 3
    x = rng.standard_normal((M, K)).astype(np.float32)
    ws = [(rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32) for _ in range(P)]
    bs = [(rng.standard_normal(N) * 0.1).astype(np.float32) for _ in range(P)]
    nb = pb.NetBuilder("siblings", device_type=1)
    nb.external_input("x", pb.K_FLOAT)
    nb.arg("pack_sibling_gemms", 0)  # keep the in-net packing out of it: this test is about the offline pass
    for p in range(P):
        nb.constant("w%d" % p, ws[p])
        nb.constant("b%d" % p, bs[p])
    for p in range(P):
        nb.op("Gemm", ["x", "w%d" % p, "b%d" % p], ["y%d" % p])
    nb.op("Concat", ["y%d" % p for p in range(P)], ["out"], axis=1)
    nb.external_output("out", pb.K_FLOAT)
    raw, opt = str(tmp_path / "raw.blaze"), str(tmp_path / "opt.blaze")
    open(raw, "wb").write(pb.convert_netdef(nb.text().encode(), True, False))
    pb.optimize_blaze(raw, opt, True)
    outs = {}
    for path in (raw, opt):
        pm = pb.PredictorManager()
        pm.load_model(path)
        p = pm.create_predictor(1, 0)
        p.reshape_input("x", [M, K])
        p.feed("x", x)
        p.register_observers(["profile"])
        p.forward()
        outs[path] = p.output_asnumpy("out").copy()
        ev = [e for e in json.loads(p.dump_observers()["profile"])["traceEvents"] if e["dur"] > 0]
        kinds = [e["name"].split(":")[0] for e in ev if not e["name"].startswith("ConstantFill")]
        if path == opt:
            assert kinds == ["FusedParallelGemm", "Split", "Concat"], kinds
            assert [e["args"]["launches"] for e in ev if e["name"].split(":")[0] in ("FusedParallelGemm", "Split")] == [1, 0]
        else:
            assert kinds == ["Gemm"] * P + ["Concat"], kinds
    want = np.concatenate([oracle.gemm_op(x, ws[p], bs[p], False, False, 1.0, 1.0) for p in range(P)], axis=1)
    np.testing.assert_allclose(outs[raw], want, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(outs[opt], want, rtol=1e-5, atol=1e-6)
    # the reference's fixture: constants only, placed on the device
    text = open(os.path.join(ROOT, "tests", "golden", "pattern", "parallel_gemm_fusion.blaze")).read().replace("device_type: 0", "device_type: 1")
    raw2, opt2 = str(tmp_path / "raw2.blaze"), str(tmp_path / "opt2.blaze")
    open(raw2, "w").write(text)
    pb.optimize_blaze(raw2, opt2, False)
    got = []
    for path in (raw2, opt2):
        pm = pb.PredictorManager()
        pm.load_model(path)
        p = pm.create_predictor(1, 0)
        p.forward()
        got.append(p.output_asnumpy("output").copy())
    a = np.arange(6, dtype=np.float32).reshape(2, 3)
    w = np.arange(6, dtype=np.float32).reshape(3, 2)
    assert np.array_equal(got[0], np.concatenate([a @ w, a @ w], axis=1)) and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_sibling_gemms_run_as_one_launch(pb, oracle, dtype):
    """Three towers read the same input: Gemm + PRelu each with weights of one shape (what the reference's ParallelGemm
    fusion rewrites into FusedParallelGemm + Split, parallel_gemm_fusion_pattern_impl.cc:20-98), plus a fourth Gemm of
    another width that must stay on its own.  By default the three run as one launch and their outputs are views of
    one buffer; with pack_sibling_gemms: 0 each runs by itself.  Both against the oracle; a second request with another
    batch size reuses the stacked weights."""
    rng = np.random.default_rng(41)
    code = pb.K_FLOAT16 if dtype == np.float16 else pb.K_FLOAT
    K, N, N4 = 48, 24, 40
    r = (lambda x: np.asarray(x, np.float32).astype(np.float16).astype(np.float32)) if dtype == np.float16 else (lambda x: np.asarray(x, np.float32))
    ws = [(rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32) for _ in range(3)]
    bs = [(rng.standard_normal(N) * 0.1).astype(np.float32) for _ in range(3)]
    slopes = [rng.uniform(0.1, 0.4, N).astype(np.float32) for _ in range(3)]
    w4 = (rng.standard_normal((K, N4)) / np.sqrt(K)).astype(np.float32)
    outs = {}
    for pack in (1, 0):
        nb = pb.NetBuilder("towers", device_type=1)
        nb.external_input("x", code)
        nb.external_output("y", code)
        nb.arg("pack_sibling_gemms", pack)
        for t in range(3):
            nb.constant("w%d" % t, ws[t], dtype=code)
            nb.constant("b%d" % t, bs[t], dtype=code)
            nb.constant("s%d" % t, slopes[t], dtype=code)
        nb.constant("w4", w4, dtype=code)
        for t in range(3):
            nb.op("Gemm", ["x", "w%d" % t, "b%d" % t], ["h%d" % t])
            nb.op("PRelu", ["h%d" % t, "s%d" % t], ["t%d" % t])
        nb.op("Gemm", ["x", "w4"], ["t3"])
        nb.op("Concat", ["t0", "t1", "t2", "t3"], ["y"], axis=1)
        pm = pb.PredictorManager()
        pm.load_model_from_string(nb.text(), True)
        p = pm.create_predictor(1, 0)
        p.register_observers(["profile"])
        got = []
        for batch in (70, 33, 70):
            x = rng.standard_normal((batch, K)).astype(np.float32) if pack == 1 or True else None
            x = np.random.default_rng(batch).standard_normal((batch, K)).astype(np.float32)
            p.reshape_input("x", x.shape)
            p.feed("x", x.astype(dtype))
            print("sibling case dtype=%s pack=%d batch=%d" % (dtype.__name__, pack, batch), flush=True)
            p.forward()
            got.append((x, p.output_asnumpy("y").astype(np.float32)))
        ev = json.loads(p.dump_observers()["profile"])["traceEvents"]
        gemms = [e for e in ev if e["name"].startswith("Gemm") and e["dur"] > 0]
        if pack:
            assert len(gemms) == 2 and sorted(e["args"]["launches"] for e in gemms) == [1, 1], gemms
        else:
            assert len(gemms) == 4
        outs[pack] = got
    tol = 2e-3 if dtype == np.float16 else 1e-5
    for pack in (1, 0):
        for x, y in outs[pack]:
            xr = r(x)
            want = [oracle.prelu(r(oracle.gemm_op(xr, r(ws[t]), r(bs[t]))), r(slopes[t])) for t in range(3)]
            want.append(oracle.gemm_op(xr, r(w4), None))
            want = r(np.concatenate([r(w_) for w_ in want], axis=1))
            assert y.shape == want.shape
            np.testing.assert_allclose(y, want, rtol=tol, atol=tol)
    for (x1, y1), (x0, y0) in zip(outs[1], outs[0]):
        np.testing.assert_allclose(y1, y0, rtol=tol, atol=tol)


def test_folded_gemm_chain_gives_the_same_outputs(pb, oracle, tmp_path):
    """Blaze_OptimizeBlaze folds Gemm(transB, alpha, beta, bias) -> Gemm(bias) with nothing between them into one Gemm on
    the product of the weights; the folded model gives the original's outputs (to the reassociation of fp32 sums) with one
    FC launch instead of two.  Also the reference's four fixtures (tests/golden/pattern/in_order_gemm_gemm_fusion*.blaze,
    constants only, moved to the device): the folded nets' outputs are those of the unfolded ones."""
    import json
    rng = np.random.default_rng(12)
    M, K, H, N = 41, 24, 32, 16
    x = rng.standard_normal((M, K)).astype(np.float32)
    w0 = (rng.standard_normal((H, K)) / np.sqrt(K)).astype(np.float32)   # used transposed
    w1 = (rng.standard_normal((H, N)) / np.sqrt(H)).astype(np.float32)
    b0, b1 = (rng.standard_normal(H) * 0.1).astype(np.float32), (rng.standard_normal(N) * 0.1).astype(np.float32)
    nb = pb.NetBuilder("chain", device_type=1)
    nb.external_input("x", pb.K_FLOAT)
    for name, v in (("w0", w0), ("b0", b0), ("w1", w1), ("b1", b1)):
        nb.constant(name, v)
    nb.op("Gemm", ["x", "w0", "b0"], ["h"], transB=1, alpha=0.5, beta=2.0)
    nb.op("Gemm", ["h", "w1", "b1"], ["out"])
    nb.external_output("out", pb.K_FLOAT)
    raw, opt = str(tmp_path / "raw.blaze"), str(tmp_path / "opt.blaze")
    open(raw, "wb").write(pb.convert_netdef(nb.text().encode(), True, False))
    pb.optimize_blaze(raw, opt, True)
    outs = {}
    for path in (raw, opt):
        pm = pb.PredictorManager()
        pm.load_model(path)
        p = pm.create_predictor(1, 0)
        p.reshape_input("x", [M, K])
        p.feed("x", x)
        p.register_observers(["profile"])
        p.forward()
        outs[path] = p.output_asnumpy("out").copy()
        ev = [e for e in json.loads(p.dump_observers()["profile"])["traceEvents"] if e["dur"] > 0]
        kinds = [e["name"].split(":")[0] for e in ev if not e["name"].startswith("ConstantFill")]
        assert kinds == (["Gemm"] if path == opt else ["Gemm", "Gemm"]), kinds
    want = oracle.gemm_op(oracle.gemm_op(x, w0, b0, False, True, 0.5, 2.0), w1, b1, False, False, 1.0, 1.0)
    np.testing.assert_allclose(outs[raw], want, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(outs[opt], want, rtol=1e-5, atol=1e-5)
    for case in ("", "2", "3", "4"):
        text = open(os.path.join(ROOT, "tests", "golden", "pattern", "in_order_gemm_gemm_fusion%s.blaze" % case)).read()
        raw2, opt2 = str(tmp_path / ("raw%s.blaze" % case)), str(tmp_path / ("opt%s.blaze" % case))
        open(raw2, "w").write(text.replace("device_type: 0", "device_type: 1"))
        pb.optimize_blaze(raw2, opt2, False)
        got = []
        for path in (raw2, opt2):
            pm = pb.PredictorManager()
            pm.load_model(path)
            p = pm.create_predictor(1, 0)
            p.forward()
            got.append(p.output_asnumpy("output").copy())
        assert got[0].shape == (2, 3) and got[0].any()
        np.testing.assert_allclose(got[1], got[0], rtol=1e-6, atol=0)


@pytest.mark.parametrize("out_dtype", [np.float32, np.float16])
@pytest.mark.parametrize("with_keys", [False, True])
def test_store_get_with_host_pointers(pb, oracle, out_dtype, with_keys):
    """SparsePuller::Get in the reference's own form (blaze/store/sparse_puller.h:77-83: every pointer host memory), as
    its host Embedding operator calls it (embedding_op.cc:87): bit-identical to the oracle's QuickEmbeddingDict::Get on
    the same block; columns of no item and the columns of an unknown table keep the caller's contents; two calls in a
    row on one thread (the second smaller) reuse the staging state; calls from other threads are served too."""
    import threading
    rng = np.random.default_rng(77)
    rows, dim = 500, 12
    data = rng.standard_normal((rows, dim)).astype(np.float32)
    keys = rng.choice(1 << 40, rows, replace=False).astype(np.int64) if with_keys else None
    pm = pb.PredictorManager()
    pm.add_table("t", data, keys=keys)
    table = oracle.Table(data, keys=None if keys is None else keys.astype(np.uint64))

    def case(batch, seed):
        r = np.random.default_rng(seed)
        seg = r.integers(0, 7, batch).astype(np.int32)
        seg[r.integers(0, batch)] = 0
        nnz = int(seg.sum())
        pick = r.integers(0, rows, nnz)
        ids = (keys[pick] if with_keys else pick).astype(np.int64)
        ids[r.random(nnz) < 0.1] = (1 << 41) + 5  # unknown keys are skipped
        vals = r.standard_normal(nnz).astype(np.float32)
        return ids, seg, vals

    def run(batch, seed):
        ids, seg, vals = case(batch, seed)
        stride = 3 + dim + dim + 4 * dim + 2
        layout = [(oracle.SUM, oracle.REVERSE, 0, 3), (oracle.AVG, oracle.ORDER, 3, 3 + dim),
                  (oracle.ASSIGN, oracle.REVERSE, 4, 3 + 2 * dim)]
        sentinel = r0 = np.random.default_rng(seed + 1).standard_normal((batch, stride)).astype(np.float32)
        want = sentinel.copy()
        oracle.embed_get(table, ids, vals, seg, [(u, d, n, want, c) for u, d, n, c in layout])
        got = sentinel.astype(out_dtype)
        pm.store_get("t", ids, seg, vals, dim, [(u, d, n, got, c) for u, d, n, c in layout])
        if out_dtype == np.float32:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        else:
            # item columns: the fp32 result narrowed once (round to nearest even); the rest: the caller's halves
            item = np.zeros(stride, bool)
            item[3:3 + 6 * dim] = True
            expect = np.where(item[None, :], want, r0.astype(np.float16).astype(np.float32)).astype(np.float16)
            assert np.array_equal(got.view(np.uint16), expect.view(np.uint16))
        # unknown table: nothing is written
        keep = sentinel.astype(out_dtype)
        before = keep.copy()
        pm.store_get("no_such_table", ids, seg, vals, dim, [(u, d, n, keep, c) for u, d, n, c in layout])
        assert np.array_equal(keep.view(np.uint8), before.view(np.uint8))

    run(300, 1)
    run(37, 2)
    run(1, 3)
    errors = []

    def worker(seed):
        try:
            run(120, seed)
        except BaseException as e:  # noqa: BLE001 -- reported by the main thread
            errors.append(e)

    ts = [threading.Thread(target=worker, args=(10 + i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    # the counts must add up to the ids handed over
    ids, seg, vals = case(20, 5)
    with pytest.raises(pb.BlazeError):
        pm.store_get("t", ids, seg, vals, dim, [(oracle.SUM, 0, 0, np.zeros((20, 4), np.float32), 0)])  # stride < dim


def _in_place_net(pb):
    """x -> Sigmoid -> x: the input is the output"""
    nb = pb.NetBuilder("in_place", device_type=1)
    nb.external_input("x", 1)
    nb.op("Sigmoid", ["x"], ["x"])
    nb.external_output("x", 1)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    return pm


def _sigmoid(x):
    return 1.0 / (1.0 + np.exp(-x.astype(np.float64)))


def test_output_after_an_in_place_input_was_reshaped(pb):
    """Forward copies an output that was read before ahead of the next Output; an input that is that output may be
    reshaped in between, and Output then answers for the new shape: the tensor's own memory, not the copy of the old
    size.  A shape beyond the fed slice is refused, as Forward refuses it."""
    rng = np.random.default_rng(3)
    pm = _in_place_net(pb)
    p = pm.create_predictor(1, 0)
    big, small = rng.standard_normal((8, 32)).astype(np.float32), rng.standard_normal((2, 32)).astype(np.float32)
    p.feed("x", big)
    p.forward()
    np.testing.assert_allclose(p.output_asnumpy("x"), _sigmoid(big), rtol=1e-5)
    want = _sigmoid(big)
    for step in range(3):  # from the second pass on the output has been copied ahead
        p.feed("x", small + step)
        p.forward()
        if step < 2:
            np.testing.assert_allclose(p.output_asnumpy("x"), _sigmoid(small + step), rtol=1e-5)
    want[:2] = _sigmoid(small + 2)
    p.reshape_input("x", big.shape)
    np.testing.assert_allclose(p.output_asnumpy("x"), want, rtol=1e-5)  # the last small pass, behind it what the large one left
    p.feed_many(p.feed_batch([("x", big)]))
    p.forward()
    p.reshape_input("x", (1000, 1000))
    with pytest.raises(pb.BlazeError, match="Output x failed"):
        p.output_asnumpy("x")


class _DeviceArray:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=3, strides=None)


@pytest.mark.parametrize("through", ["output", "in-place input", "input under a Reshape"])
@pytest.mark.parametrize("when", ["before the first pass", "after a copy ahead"])
def test_output_sees_what_was_written_through_a_device_address(pb, through, when):
    """Output returns the tensor as it is when Output is called, also where the caller changed it in place after Forward
    through an address from output_device_ptr or input_device_ptr -- on every pass, whether the address was taken
    before the first pass or after Forward had already copied an output ahead."""
    import torch
    nb = pb.NetBuilder("addr", device_type=1)
    nb.external_input("x", 1)
    if through == "in-place input":
        nb.op("Sigmoid", ["x"], ["x"])
        out = "x"
    elif through == "input under a Reshape":
        nb.constant("shape", np.array([16, 4], np.int32))
        nb.op("Reshape", ["x", "shape"], ["y"])
        out = "y"
    else:
        nb.op("Sigmoid", ["x"], ["y"])
        out = "y"
    nb.external_output(out, 1)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    x = np.random.default_rng(4).standard_normal((4, 16)).astype(np.float32)

    def address():
        return p.output_device_ptr(out) if through == "output" else p.input_device_ptr("x")

    p.feed("x", x)
    p.forward()
    if when == "after a copy ahead":
        for _ in range(2):
            p.output_asnumpy(out)
            p.forward()
    for step in range(4):
        view = torch.as_tensor(_DeviceArray(address(), x.shape), device="cuda")
        view.fill_(float(step))
        torch.cuda.synchronize()
        got = p.output_asnumpy(out)
        assert got.size == x.size and (got == step).all(), (step, got.reshape(-1)[:4])
        p.forward()
        if through == "output":
            np.testing.assert_allclose(p.output_asnumpy(out), _sigmoid(x), rtol=1e-5)
        elif through == "in-place input":
            np.testing.assert_allclose(p.output_asnumpy(out), _sigmoid(np.full_like(x, step)), rtol=1e-5)


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_outputs_with_every_bit_set_arrive_too(pb, dtype):
    """A pass ends when its outputs have reached the host, which shows in the value that stood there before (all bits set): an
    output that holds that value comes out as any other, in the passes before and behind it too."""
    nb = pb.NetBuilder("bits", device_type=1)
    code = pb.K_FLOAT16 if dtype == np.float16 else pb.K_FLOAT
    for name in ("a", "b"):
        nb.external_input(name, code)
    nb.op("Concat", ["a", "b"], ["y"], axis=1)
    nb.external_output("y", code)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    rng = np.random.default_rng(9)
    bits = np.uint32 if dtype == np.float32 else np.uint16
    for step in range(80):  # (every 32nd pass waits for the stream)
        a, b = rng.standard_normal((5, 3)).astype(dtype), rng.standard_normal((5, 4)).astype(dtype)
        if step in (3, 4, 40):
            b.view(bits)[step % 5, step % 4] = ~bits(0)
        p.reshape_input("a", a.shape)
        p.reshape_input("b", b.shape)
        p.feed_many(p.feed_batch([("a", a), ("b", b)]))
        p.forward()
        got = p.output_asnumpy("y").reshape(5, 7)
        assert np.array_equal(got.view(bits), np.concatenate([a.view(bits), b.view(bits)], 1)), step


def _in_another_thread(f):
    import threading
    result = []
    t = threading.Thread(target=lambda: result.append(f()))
    t.start()
    t.join()
    return result[0]


@pytest.mark.parametrize("what", ["feed", "feed_many", "launch", "device address"])
def test_another_threads_work_waits_for_a_pass_that_ended_by_its_outputs(pb, what):
    """A pass may end when its outputs are on the host, the end of its last launch still running on this thread's stream.  What
    another thread queues, on a stream of its own, comes behind that."""
    nb = pb.NetBuilder("arrived", device_type=1)
    nb.external_input("x", pb.K_FLOAT)
    nb.op("Sigmoid", ["x"], ["y"])
    nb.external_output("y", pb.K_FLOAT)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    x = np.random.default_rng(2).standard_normal((4, 16)).astype(np.float32)
    do = {"feed": lambda: p.feed("x", x), "feed_many": lambda: p.feed_many(p.feed_batch([("x", x)])), "launch": p.forward_launch,
          "device address": lambda: p.output_device_ptr("y")}[what]

    def state():
        return p.dump_observers()["pass"]

    def there():
        do()
        now = state()
        if what == "launch":
            p.forward_wait()
        return now

    seen = 0
    for _ in range(16):
        p.feed("x", x)
        p.forward()
        np.testing.assert_allclose(p.output_asnumpy("y").reshape(4, 16), _sigmoid(x), rtol=1e-5)
        if state() != "arrived":  # (the first pass, and one in which this thread was interrupted)
            continue
        seen += 1
        p.feed("x", x)
        assert state() == "arrived"  # (the same stream)
        assert _in_another_thread(there) == "ended"
        p.forward()
        np.testing.assert_allclose(p.output_asnumpy("y").reshape(4, 16), _sigmoid(x), rtol=1e-5)
        if what == "device address":
            assert state() == "ended"
            break
    assert seen > 0


@pytest.mark.parametrize("declared", [("y", ), ("y", "z")])
def test_a_pass_ends_by_its_outputs_only_where_every_operator_feeds_one(pb, declared):
    """Operators behind the last output, which nothing shows the end of: such a net's stream is waited for."""
    nb = pb.NetBuilder("tail", device_type=1)
    nb.external_input("x", pb.K_FLOAT)
    nb.op("Sigmoid", ["x"], ["y"])
    nb.op("Sigmoid", ["x"], ["t"])
    nb.op("Sigmoid", ["t"], ["z"])
    for o in declared:
        nb.external_output(o, pb.K_FLOAT)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    x = np.random.default_rng(2).standard_normal((4, 16)).astype(np.float32)
    states = set()
    for _ in range(8):
        p.feed("x", x)
        p.forward()
        states.add(p.dump_observers()["pass"])
        for o in declared:
            p.output_asnumpy(o)
    assert ("arrived" in states) == (len(declared) == 2), states


def test_feed_forward_and_output_in_threads_of_their_own(pb):
    """Inputs fed by one thread, the pass run by another, the output read by a third, each of them new or the same as last time,
    fed twice before a pass, read twice behind it, and through the device address: always the pass's own."""
    import threading
    import torch
    nb = pb.NetBuilder("threads", device_type=1)
    nb.external_input("x", pb.K_FLOAT)
    rng = np.random.default_rng(10)
    w, u = (rng.standard_normal(sh).astype(np.float32) for sh in ((64, 32), (32, 2)))
    nb.constant("w", w)
    nb.constant("u", u)
    nb.op("Gemm", ["x", "w"], ["h"])
    nb.op("Gemm", ["h", "u"], ["y"])
    nb.external_output("y", pb.K_FLOAT)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    errors = []

    def run(where, f):
        def guarded():
            try:
                f()
            except Exception as e:  # noqa: BLE001
                errors.append(repr(e))
        if where == "here":
            return guarded()
        t = threading.Thread(target=guarded)
        t.start()
        t.join()

    for step in range(60):
        x = rng.standard_normal((300, 64)).astype(np.float32)
        want = x.astype(np.float64) @ w.astype(np.float64) @ u.astype(np.float64)
        who = ["here" if rng.random() < 0.6 else "there" for _ in range(3)]
        p.reshape_input("x", x.shape)
        if step % 7 == 0:
            run(who[2], lambda: p.feed_many(p.feed_batch([("x", x + 1)])))
        if step % 3:
            run(who[0], lambda: p.feed_many(p.feed_batch([("x", x)])))
        else:
            run(who[0], lambda: p.feed("x", x))
        run(who[1], p.forward)
        got = []
        run(who[2], lambda: got.append(p.output_asnumpy("y").copy()))
        if step % 5 == 0:
            run(who[0], lambda: got.append(p.output_asnumpy("y").copy()))
        if step > 50:
            got.append(torch.as_tensor(_DeviceArray(p.output_device_ptr("y"), (300, 2)), device="cuda").cpu().numpy())
        assert not errors, errors
        for g in got:
            np.testing.assert_allclose(g.reshape(300, 2), want, rtol=0, atol=2e-4, err_msg="step %d %s" % (step, who))


def test_outputs_copied_ahead_of_output(pb):
    """Ten outputs (one launch copies eight ahead) at batches whose outputs are below and above what is copied ahead
    (64 KB): read once, twice or not at all after a pass, in either order, after growing and shrinking.  Every read is the
    pass's own result, and from the second pass of a shape on neither Forward nor Output allocates."""
    rng = np.random.default_rng(6)
    nb = pb.NetBuilder("many", device_type=1)
    nb.external_input("x", 1)
    cs = [np.float32(0.5 * k - 2.0) for k in range(10)]
    for k, c in enumerate(cs):
        nb.constant("c%d" % k, np.full((1, 8), c, np.float32))
        nb.op("Add", ["x", "c%d" % k], ["y%d" % k])
        nb.external_output("y%d" % k, 1)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    for batch in (3, 2048, 2049, 1, 700):  # 2048 rows of 32 bytes are 64 KB
        for step, reads in enumerate(((0, 1, 2), range(10), range(9, -1, -1), (9, 9, 8), (), tuple(range(10)) * 2, (4, 4, 4))):
            x = rng.standard_normal((batch, 8)).astype(np.float32)
            p.feed("x", x)
            if step == 2:
                before = pb.allocation_count()  # every output of this shape has been read once
            p.forward()
            for k in reads:
                np.testing.assert_array_equal(p.output_asnumpy("y%d" % k), x + cs[k], err_msg="batch %d step %d output %d" % (batch, step, k))
        assert pb.allocation_count() == before


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("k,n,heads", [(256, 100, 2), (64, 50, 1), (128, 9, 3), (96, 255, 8), (40, 17, 1), (256, 4 * 25, 8)])
def test_head_behind_a_layer_of_any_number_of_columns(pb, dtype, k, n, heads):
    """columns that are no multiple of eight: the head in the layer's launch up to a number of rows, two launches beyond it,
    against 64 bits from the rounded layer and against two launches throughout (fuse_fc_head: 0)"""
    rng = np.random.default_rng(k + n)
    w1, b1 = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(dtype), (rng.standard_normal(n) * 0.1).astype(dtype)
    w2, b2 = (rng.standard_normal((n, heads)) / np.sqrt(n)).astype(dtype), (rng.standard_normal(heads) * 0.1).astype(dtype)
    got = {}
    rows = (1, 15, 300, 1025, (200 << 10) // k, 2048, 2049, (512 << 10) // k + 1)
    xs = [rng.standard_normal((m, k)).astype(dtype) for m in rows]
    for fuse in (1, 0):
        nb = pb.NetBuilder("any%d" % fuse, device_type=1)
        nb.arg("fuse_fc_head", fuse)
        code = pb.K_FLOAT16 if dtype == np.float16 else pb.K_FLOAT
        nb.external_input("x", code)
        for name, v in (("w1", w1), ("b1", b1), ("w2", w2), ("b2", b2)):
            nb.constant(name, v)
        nb.op("Gemm", ["x", "w1", "b1"], ["h"], transB=0)
        nb.op("Sigmoid", ["h"], ["hs"])
        nb.op("Gemm", ["hs", "w2", "b2"], ["z"], transB=0)
        nb.op("Softmax", ["z"], ["p"], axis=1)
        nb.external_output("p", code)
        pm = pb.PredictorManager()
        pm.load_model_from_string(nb.text(), True)
        p = pm.create_predictor(1, 0)
        got[fuse] = []
        for x in xs:
            p.feed("x", x)
            p.forward()
            got[fuse].append(p.output_asnumpy("p").astype(np.float64).reshape(len(x), heads))
    for x, g1, g0 in zip(xs, got[1], got[0]):
        h = _sigmoid(x.astype(np.float64) @ w1.astype(np.float64) + b1)
        e = np.exp(h @ w2.astype(np.float64) + b2)
        # fp16: h is rounded (2^-11 of at most 1, weights of 1 / sqrt(n)), and so is the result; fp32: sums of k and n terms
        tol = 4 * 2.0**-11 if dtype == np.float16 else 1e-5
        for g in (g1, g0):
            np.testing.assert_allclose(g, e / e.sum(1, keepdims=True), rtol=0, atol=tol, err_msg="%d rows" % len(x))


def _launches(p, op_type):
    ev = json.loads(p.dump_observers()["profile"])["traceEvents"]
    return sum(e["args"]["launches"] for e in ev if e["name"].split(":")[0] == op_type and e["dur"] > 0)


@pytest.mark.parametrize("dtype,k,n,rows,launches", [
    (np.float16, 256, 250, 300, 1), (np.float16, 384, 250, 2048, 1), (np.float16, 384, 250, 2049, 2), (np.float16, 400, 250, 300, 2),
    (np.float16, 512, 100, 1536, 1), (np.float16, 512, 100, 1537, 2), (np.float32, 144, 250, 300, 1), (np.float32, 400, 250, 300, 2),
    (np.float32, 400, 92, 614, 1), (np.float32, 400, 92, 615, 2), (np.float32, 400, 93, 1, 2), (np.float32, 64, 100, 2049, 2)])
def test_a_head_behind_any_columns_stays_where_it_is_faster(pb, dtype, k, n, rows, launches):
    """the lines in k * n, rows * k and rows up to which a head rides behind columns that are no multiple of eight"""
    rng = np.random.default_rng(k + n)
    w1, w2 = (rng.standard_normal((k, n)) / np.sqrt(k)).astype(dtype), (rng.standard_normal((n, 1)) / np.sqrt(n)).astype(dtype)
    code = pb.K_FLOAT16 if dtype == np.float16 else pb.K_FLOAT
    nb = pb.NetBuilder("line", device_type=1)
    nb.external_input("x", code)
    nb.external_output("z", code)
    nb.constant("w1", w1)
    nb.constant("w2", w2)
    nb.op("Gemm", ["x", "w1"], ["h"])
    nb.op("Sigmoid", ["h"], ["s"])
    nb.op("Gemm", ["s", "w2"], ["z"])
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    p.register_observers(["profile"])
    x = rng.standard_normal((rows, k)).astype(dtype)
    p.feed("x", x)
    p.forward()
    assert _launches(p, "Gemm") == launches
    want = _sigmoid(x.astype(np.float64) @ w1.astype(np.float64)) @ w2.astype(np.float64)
    # fp16: the layer's output is rounded (2^-11 of at most 1, n weights of 1 / sqrt(n) whose errors go both ways), and the result
    tol = (4 + 2 * np.abs(want).max()) * 2.0**-11 if dtype == np.float16 else 1e-5
    np.testing.assert_allclose(p.output_asnumpy("z").astype(np.float64), want, rtol=0, atol=tol)


@pytest.mark.parametrize("dtype,P,n,K,heads_in", [
    (np.float16, 2, 100, 64, 2048), (np.float16, 3, 9, 64, 2048), (np.float16, 3, 172, 256, 2048), (np.float16, 3, 220, 256, 0),
    (np.float16, 4, 100, 64, 2048), (np.float16, 4, 60, 64, 0), (np.float16, 5, 50, 64, 0), (np.float16, 6, 100, 64, 1024),
    (np.float32, 2, 50, 64, 2048), (np.float32, 2, 100, 64, 0), (np.float32, 2, 250, 48, 0), (np.float32, 3, 50, 64, 0), (np.float32, 4, 33, 64, 0)])
def test_towers_with_heads_on_one_input(pb, dtype, P, n, K, heads_in):
    """P towers K -> n -> 2 written one after the other, n no multiple of eight: up to `heads_in` rows each runs with its head as one
    launch, else the layers are one launch and each head one.  Rows below and beyond the limits in turn, against 64 bits from
    the rounded layer and against one launch for everything."""
    rng = np.random.default_rng(P * n)
    code = pb.K_FLOAT16 if dtype == np.float16 else pb.K_FLOAT
    ws = [[(rng.standard_normal(sh) / np.sqrt(sh[0])).astype(dtype) for sh in ((K, n), (1, n), (n, 2), (1, 2))] for _ in range(P)]
    xs = [rng.standard_normal((m, K)).astype(dtype) for m in (300, 4096, 1, 2049, 2048, 300)]
    got = {}
    for fuse in (1, 0):
        nb = pb.NetBuilder("towers%d" % fuse, device_type=1)
        nb.arg("fuse_fc_head", fuse)
        nb.arg("pack_sibling_gemms", fuse)
        nb.external_input("x", code)
        for t, (w, b, u, c) in enumerate(ws):
            for name, v in (("w", w), ("b", b[0]), ("u", u), ("c", c[0])):
                nb.constant("%s%d" % (name, t), v)
            nb.op("Gemm", ["x", "w%d" % t, "b%d" % t], ["h%d" % t])
            nb.op("Sigmoid", ["h%d" % t], ["s%d" % t])
            nb.op("Gemm", ["s%d" % t, "u%d" % t, "c%d" % t], ["z%d" % t])
            nb.op("Softmax", ["z%d" % t], ["p%d" % t], axis=1)
            nb.external_output("p%d" % t, code)
        pm = pb.PredictorManager()
        pm.load_model_from_string(nb.text(), True)
        p = pm.create_predictor(1, 0)
        p.register_observers(["profile"])
        got[fuse] = []
        for x in xs:
            p.feed("x", x)
            p.forward()
            got[fuse].append([p.output_asnumpy("p%d" % t).astype(np.float64) for t in range(P)])
            if fuse:
                assert _launches(p, "Gemm") == (P if len(x) <= heads_in else 1 + P), len(x)
    tol = 4 * 2.0**-11 if dtype == np.float16 else 1e-5  # (as for one tower: the rounded layer, weights of 1 / sqrt(n))
    for x, g1, g0 in zip(xs, got[1], got[0]):
        for t, (w, b, u, c) in enumerate(ws):
            h = _sigmoid(x.astype(np.float64) @ w.astype(np.float64) + b)
            e = np.exp(h @ u.astype(np.float64) + c)
            for g in (g1[t], g0[t]):
                np.testing.assert_allclose(g, e / e.sum(1, keepdims=True), rtol=0, atol=tol, err_msg="%d rows, tower %d" % (len(x), t))


@pytest.mark.parametrize("w,n", [(54, 36), (24, 9)])
def test_attention_input_in_front_of_a_layer_with_a_head(pb, w, n):
    """[q, k, q - k, q * k] -> n columns, no multiple of eight -> 1: beyond the rows that a head is in the layer's launch at, the
    layer computes its input while it loads it and the Concat's tensor is never made; below, the Concat runs and the head
    is in the launch.  Against the operators one by one."""
    import torch
    rng = np.random.default_rng(w)
    ws = {"w1": (4 * w, n), "b1": (n, ), "g": (n, ), "m": (n, ), "v": (n, ), "w2": (n, 1), "b2": (1, )}
    ws = {k: (np.abs(rng.standard_normal(sh)) + 0.5 if k == "v" else rng.standard_normal(sh) / np.sqrt(sh[0])).astype(np.float16) for k, sh in ws.items()}
    reqs = [(rng.standard_normal((B, 1, w)).astype(np.float16), rng.standard_normal((B, T, w)).astype(np.float16)) for B, T in ((600, 50), (1, 20), (683, 3), (600, 50))]
    got = {}
    for fuse in (1, 0):
        nb = pb.NetBuilder("att%d" % fuse, device_type=1)
        for switch in ("fuse_fc_head", "fuse_concat_into_fc"):
            nb.arg(switch, fuse)
        nb.external_input("q", pb.K_FLOAT16)
        nb.external_input("k", pb.K_FLOAT16)
        nb.external_output("s", pb.K_FLOAT16)
        for k, v in ws.items():
            nb.constant(k, v)
        nb.op("Sub", ["q", "k"], ["sub"])
        nb.op("Mul", ["q", "k"], ["mul"])
        nb.op("BroadcastTo", ["q", "sub"], ["bq"])
        nb.op("Concat", ["bq", "k", "sub", "mul"], ["a"], axis=2)
        nb.op("Gemm", ["a", "w1", "b1"], ["h"])
        nb.op("Dice", ["h", "g", "m", "v"], ["d"])
        nb.op("Gemm", ["d", "w2", "b2"], ["s"])
        pm = pb.PredictorManager()
        pm.load_model_from_string(nb.text(), True)
        p = pm.create_predictor(1, 0)
        p.register_observers(["profile"])
        got[fuse] = []
        for i, (q, k) in enumerate(reqs):
            p.feed("q", q)
            p.feed("k", k)
            torch.cuda.synchronize()
            free = torch.cuda.mem_get_info()[0]
            p.forward()
            if fuse and i == 0:  # the layer's own output is stored, the Concat's (at least as large) is not
                assert free - torch.cuda.mem_get_info()[0] < q.shape[0] * k.shape[1] * 4 * w * 2
            got[fuse].append(p.output_asnumpy("s").astype(np.float64))
            if fuse:
                assert _launches(p, "Gemm") == 2
    for (q, k), s1, s0 in zip(reqs, got[1], got[0]):
        assert s1.shape == (k.shape[0], k.shape[1], 1) and s1.any()
        # both round the input pieces and the layer's output alike; the layer's sums come in another order: a rounding of its
        # output of |h| of a few, times weights of 1 / sqrt(n), here and there, and one of the score
        np.testing.assert_allclose(s1, s0, rtol=0, atol=4 * 2.0**-11 * max(1.0, np.abs(s0).max()))


@pytest.mark.parametrize("touched", ["by nothing else", "read by an operator", "written in place"])
def test_outputs_that_a_layer_copies_in_its_own_launch(pb, touched):
    """A skinny layer (s) and a layer's skinny head (p) write the host's copy of their outputs themselves, up to 64 KB, as the
    observers' dump says: read after every pass, some passes or twice, at growing and shrinking batches; and where another operator of the net reads or
    overwrites the output, which is then copied as it is in the end."""
    rng = np.random.default_rng(16)
    w1, w2, w3 = (rng.standard_normal(s).astype(np.float32) * 0.3 for s in ((40, 16), (16, 2), (40, 3)))
    nb = pb.NetBuilder("copies", device_type=1)
    nb.external_input("x", 1)
    for k, w in (("w1", w1), ("w2", w2), ("w3", w3)):
        nb.constant(k, w)
    nb.op("Gemm", ["x", "w1"], ["h"], transB=0)
    nb.op("Sigmoid", ["h"], ["hs"])
    nb.op("Gemm", ["hs", "w2"], ["z"], transB=0)
    nb.op("Softmax", ["z"], ["p"], axis=1)
    nb.op("Gemm", ["x", "w3"], ["s"], transB=0)
    outs = ["p", "s"]
    if touched == "read by an operator":
        nb.op("Sigmoid", ["s"], ["s2"])
        nb.op("Sigmoid", ["p"], ["p2"])
        outs += ["p2", "s2"]
    elif touched == "written in place":
        nb.constant("one", np.ones((1, 3), np.float32))
        nb.op("Add", ["s", "one"], ["s"])
    for o in outs:
        nb.external_output(o, 1)
    shared = {"by nothing else": "", "read by an operator": "ps", "written in place": "s"}[touched]
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    for batch in (1, 300, 5461, 5462, 8192, 8193, 7):  # 64 KB are 8192 rows of p, 5461 of s
        for step in range(5):
            x = rng.standard_normal((batch, 40)).astype(np.float32)
            p.feed("x", x)
            p.forward()
            where = json.loads(p.dump_observers()["outputs"])
            # (step 0: what Output made for another batch; step 3: s was not read after the pass before)
            for o, cols in (("p", 2), ("s", 3)) if step else ():
                by = "operator" if o not in shared else "copied"
                expect = "device" if batch * cols * 4 > 64 << 10 or (step == 3 and o == "s") else by
                assert where[o] == expect, "batch %d step %d %s" % (batch, step, o)
            d = x.astype(np.float64)
            e = np.exp(_sigmoid(d @ w1) @ w2)
            want = {"p": e / e.sum(1, keepdims=True), "s": d @ w3 + (touched == "written in place")}
            want.update(p2=_sigmoid(want["p"]), s2=_sigmoid(want["s"]))
            for o in (outs if step != 2 else outs[:1]) + (outs[:1] if step == 3 else []):
                np.testing.assert_allclose(p.output_asnumpy(o), want[o], rtol=1e-5, atol=1e-5, err_msg="batch %d step %d %s" % (batch, step, o))


def test_the_pass_after_the_first_output_allocates_nothing(pb):
    """The buffer that Forward copies an output into is made by Output, not between a launch and its wait."""
    pm = _in_place_net(pb)
    p = pm.create_predictor(1, 0)
    x = np.random.default_rng(8).standard_normal((5, 7)).astype(np.float32)
    p.feed("x", x)
    p.forward()
    np.testing.assert_allclose(p.output_asnumpy("x"), _sigmoid(x), rtol=1e-5)
    before = pb.allocation_count()
    for _ in range(3):
        p.feed("x", x)
        p.forward()
        np.testing.assert_allclose(p.output_asnumpy("x"), _sigmoid(x), rtol=1e-5)
    assert pb.allocation_count() == before


@pytest.mark.parametrize("n_in", [1, 8, 9, 17])
def test_feed_many_of_strided_inputs(pb, n_in):
    """Inputs that live side by side inside a Concat's output: one launch takes eight of them.  Odd widths, a plain input
    beside them, an input named twice (the last one counts), a batch that grows and shrinks."""
    rng = np.random.default_rng(n_in)
    nb = pb.NetBuilder("strided", device_type=1)
    widths = [1 + (5 * k) % 7 for k in range(n_in)]
    for k in range(n_in):
        nb.external_input("x%d" % k, 1)
    nb.external_input("plain", 1)
    nb.op("Concat", ["x%d" % k for k in range(n_in)], ["z"], axis=1)
    nb.op("Sigmoid", ["plain"], ["s"])
    nb.external_output("z", 1)
    nb.external_output("s", 1)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    for batch in (4, 301, 2):
        for _ in range(2):
            xs = [rng.standard_normal((batch, w)).astype(np.float32) for w in widths]
            plain = rng.standard_normal((batch, 3)).astype(np.float32)
            items = [("x%d" % k, a) for k, a in enumerate(xs)] + [("plain", plain)]
            for name, a in items:
                p.reshape_input(name, a.shape)
            p.feed_many(p.feed_batch([("x0", xs[0] + 1)] + items))
            p.forward()
            np.testing.assert_array_equal(p.output_asnumpy("z"), np.concatenate(xs, 1))
            np.testing.assert_allclose(p.output_asnumpy("s"), _sigmoid(plain), rtol=1e-5)


# bytes of the inputs, one behind the other on multiples of 256: parts end after 384, 960, 1824 KB and then every MB, from 4 MB on there
# are as many even ones as whole MB, unless less than half a part would be left
@pytest.mark.parametrize("sizes", [[4, 393212], [393216, 196604], [393216, 196608], [393216, 196612], [393000, 300, 300000],   # in the padding; left over: half a part or less
                                   [393212, 4, 600000], [983040, 4, 430000], [300, 983040 - 512, 900000, 2 << 20], [(4 << 20) - 256, 4],
                                   [(4 << 20) - 512, 252], [5 << 20, 260], [(1 << 20) - 4, 4, 4 << 20]])
def test_feed_many_at_the_borders_of_its_parts(pb, sizes):
    rng = np.random.default_rng(sum(sizes))
    nb = pb.NetBuilder("parts", device_type=1)
    for k in range(len(sizes)):
        nb.external_input("x%d" % k, pb.K_FLOAT)
        nb.op("Sigmoid", ["x%d" % k], ["y%d" % k])
        nb.external_output("y%d" % k, pb.K_FLOAT)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    for _ in range(2):
        xs = [rng.standard_normal((s // 4, 1)).astype(np.float32) for s in sizes]
        for k, x in enumerate(xs):
            p.reshape_input("x%d" % k, x.shape)
        p.feed_many(p.feed_batch([("x%d" % k, x) for k, x in enumerate(xs)]))
        p.forward()
        for k, x in enumerate(xs):
            np.testing.assert_allclose(p.output_asnumpy("y%d" % k).reshape(-1), _sigmoid(x).reshape(-1), rtol=1e-5)


# 64-bit ids cross as their lower halves and equal 32-bit words as one, in blocks of 256 words: the word that does not fit stands at
# the edges of blocks and parts, at the end, or nowhere
@pytest.mark.parametrize("n,odd", [(1, []), (255, []), (256, []), (1023, [1022]), (1024, []), (1025, [1024]), (5000, [7]), (5000, [8]), (5000, [1023]),
                                   (5000, [1024]), (5000, [4999]), (5000, [2048, 3000]), (49152, [49151]), (49153, [49152]), (200001, [131072]), (700000, [])])
def test_feed_many_of_words_that_are_packed(pb, n, odd):
    import torch
    rng = np.random.default_rng(n)
    nb = pb.NetBuilder("packed", device_type=1)
    kinds = {"ids": pb.K_INT64, "before": pb.K_FLOAT, "values": pb.K_FLOAT, "counts": pb.K_INT32, "more": pb.K_INT64}
    nb.constant("flat", np.array([-1], np.int32))
    for name, code in kinds.items():
        nb.external_input(name, code)
        nb.op("Reshape", [name, "flat"], ["flat_" + name])
        nb.external_output("flat_" + name, code)
    nb.external_input("x", pb.K_FLOAT)
    nb.op("Sigmoid", ["x"], ["y"])
    nb.external_output("y", pb.K_FLOAT)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    for turn in range(3):
        ids = rng.integers(0, 1 << 32, n, dtype=np.int64)
        more = rng.integers(-1 << 62, 1 << 62, n // 3 + 1, dtype=np.int64)
        values, counts = np.full(n, -0.0 if turn else np.nan, np.float32), np.full(n, 255, np.int32)
        for k in odd if turn < 2 else []:
            ids[k] = -1 - k if turn else ids[k] + (1 << 32)
            values[k], counts[k] = 0.0 if turn else 1.0, -255
        feed = {"ids": ids, "before": rng.standard_normal(67).astype(np.float32), "values": values, "counts": counts, "more": more, "x": values[:3].copy()}
        for name, a in feed.items():
            p.reshape_input(name, a.shape)
        p.feed_many(p.feed_batch(list(feed.items())))
        p.forward()
        for name in kinds:
            there = dict(shape=feed[name].shape, typestr=feed[name].dtype.str, data=(p.input_device_ptr(name), False), version=3, strides=None)
            got = torch.as_tensor(type("View", (), dict(__cuda_array_interface__=there))(), device="cuda").cpu().numpy()
            assert got.tobytes() == feed[name].tobytes(), (turn, name)


# the line from which a request is packed, and the edges of the first blocks
@pytest.mark.parametrize("n,odd", [(4095, []), (4096, []), (4097, [255]), (5000, [255]), (5000, [256]), (5000, [511]), (5000, [513])])
def test_feed_many_packed_or_not(pb, n, odd):
    test_feed_many_of_words_that_are_packed(pb, n, odd)


@pytest.mark.parametrize("lists", [21, 22, 30])  # 63 and 66 ranges, where a launch takes 64, and 90
def test_feed_many_of_more_ranges_than_a_launch_takes(pb, lists):
    """lists of ids and equal values with short counts between them, every third value differing somewhere: each input arrives as it is"""
    import torch
    rng = np.random.default_rng(lists)
    nb = pb.NetBuilder("ranges", device_type=1)
    nb.constant("flat", np.array([-1], np.int32))
    kinds = {}
    for i in range(lists):
        kinds.update({"ids%d" % i: pb.K_INT64, "values%d" % i: pb.K_FLOAT, "counts%d" % i: pb.K_INT32})
    for name, code in kinds.items():
        nb.external_input(name, code)
        nb.op("Reshape", [name, "flat"], ["flat_" + name])
        nb.external_output("flat_" + name, code)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    p = pm.create_predictor(1, 0)
    for turn in range(2):
        feed = {}
        for i in range(lists):
            n = 1600 + 37 * i  # 12.8 and 6.4 KB on: 22 lists are one part
            feed["ids%d" % i] = rng.integers(0, 1 << 32, n, dtype=np.int64)
            feed["values%d" % i] = np.full(n, 1 + i, np.float32)
            feed["counts%d" % i] = rng.integers(0, 20, 201).astype(np.int32)
            if turn and i % 3 == 0:
                feed["values%d" % i][rng.integers(n)] = -1
        for name, a in feed.items():
            p.reshape_input(name, a.shape)
        p.feed_many(p.feed_batch(list(feed.items())))
        p.forward()
        for name in kinds:
            there = dict(shape=feed[name].shape, typestr=feed[name].dtype.str, data=(p.input_device_ptr(name), False), version=3, strides=None)
            got = torch.as_tensor(type("View", (), dict(__cuda_array_interface__=there))(), device="cuda").cpu().numpy()
            assert got.tobytes() == feed[name].tobytes(), (turn, name)


def _tower(pb, ws, bs, acts, chain, heads):
    kind = pb.K_FLOAT if ws[0].dtype == np.float32 else pb.K_FLOAT16
    nb = pb.NetBuilder("tower%d" % chain, device_type=1)
    nb.arg("chain_narrow_fcs", chain)
    nb.external_input("x", kind)
    params = [[] if a is None else a[1:] for a in acts]
    for i, (w, b) in enumerate(zip(ws, bs)):  # (in front of the layers: operators are joined where they follow each other)
        nb.constant("w%d" % i, w)
        nb.constant("b%d" % i, b)
        for j, p in enumerate(params[i] if i < 2 else []):
            nb.constant("a%d%d" % (i, j), p)
    h = "x"
    for i in range(3):
        nb.op("Gemm", [h, "w%d" % i, "b%d" % i], ["g%d" % i], transB=0)
        h = "g%d" % i
        if i < 2 and acts[i] is not None:
            nb.op(acts[i][0], [h] + ["a%d%d" % (i, j) for j in range(len(params[i]))], ["h%d" % i])
            h = "h%d" % i
    if heads > 1:
        nb.op("Softmax", [h], ["p"], axis=1)
    else:
        nb.op("Sigmoid", [h], ["p"])
    nb.external_output("p", kind)
    pm = pb.PredictorManager()
    pm.load_model_from_string(nb.text(), True)
    return pm.create_predictor(1, 0)


def _tower_pays(rows, k, n1, n2):
    weights = k * n1 + n1 * n2
    return rows <= 4096 and k <= 1280 and (rows >= 1200 and k <= 1024 or weights <= (256 if k <= 768 or rows >= 600 and k <= 1024 else 144) << 10)


def _tower_launches(p):
    layers = [e for e in json.loads(p.dump_observers()["profile"])["traceEvents"] if e["name"].startswith("Gemm:")][:2]
    return sum(e["args"]["launches"] for e in layers), [e["dur"] for e in layers]


def _tower_act(z, act):
    if act is None:
        return z
    if act[0] == "PRelu":
        return np.where(z > 0, z, z * act[1].astype(np.float64))
    if act[0] == "Dice":
        g, m, v = (a.astype(np.float64) for a in act[1:])
        p = _sigmoid((z - m) / np.sqrt(v + 1e-8))
        return (1 - p) * g * z + p * z
    return _sigmoid(z)


# k: one input, rows of 16-byte, 4-byte and 2-byte steps, whole and ragged 64s, the longest that is staged at once and the longest taken;
# n1: one and two blocks a wave; n2, heads: the smallest and the largest; rows: one workgroup's edges and the lines of bz::fc_tower_pays
@pytest.mark.parametrize("k,n1,n2,heads,rows", [(1, 9, 9, 1, (1, 33)), (64, 32, 33, 2, (31, 32, 33, 4096, 4097)), (65, 33, 64, 8, (5, 300)), (66, 256, 100, 2, (300, 64)),
                                                (445, 256, 100, 2, (300, 1, 2049)), (448, 257, 256, 3, (40, 4096)), (1024, 192, 96, 1, (70, 1301)), (1027, 104, 40, 2, (33, 500)),
                                                (1280, 88, 40, 2, (300, )), (896, 512, 256, 2, (1199, 1200, 2048, 32)), (128, 512, 250, 8, (77, 1500))])
@pytest.mark.parametrize("act", ["PRelu", "Dice", "Sigmoid", None])
def test_tower_in_one_launch(pb, k, n1, n2, heads, rows, act):
    """fp16 layer -> layer -> skinny layer against 64 bits from the rounded layers and against one launch a layer, the rows growing and
    shrinking past the lines beyond which it is no launch of its own; and while the operators are timed one by one."""
    rng = np.random.default_rng(k * n1 + n2)
    sizes = (k, n1, n2, heads)
    ws = [(rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float16) for s in zip(sizes, sizes[1:])]
    bs = [(rng.standard_normal(n) * 0.1).astype(np.float16) for n in sizes[1:]]
    acts = []
    for n in (n1, n2):
        p = [rng.uniform(0.1, 0.4, n).astype(np.float16), (rng.standard_normal(n) * 0.1).astype(np.float16), rng.uniform(0.5, 1.5, n).astype(np.float16)]
        acts.append({"PRelu": ("PRelu", p[0]), "Dice": ("Dice", *p), "Sigmoid": ("Sigmoid", ), None: None}[act])
    one, apart = (_tower(pb, ws, bs, acts, chain, heads) for chain in (1, 0))
    for step, m in enumerate(rows + rows[:1]):
        print("tower %d x %d -> %d -> %d -> %d %s" % (m, k, n1, n2, heads, act), flush=True)
        if step == len(rows):
            one.register_observers(["profile"])
        x = rng.standard_normal((m, k)).astype(np.float16)
        got = []
        for p in (one, apart):
            p.feed("x", x)
            p.forward()
            got.append(p.output_asnumpy("p").astype(np.float64).reshape(m, heads))
        # (a head behind columns that are no multiple of eight may be a launch of its own; two layers with nothing between are made one)
        if act is not None and step < len(rows):
            assert (_tower_launches(one)[0] == 1) == _tower_pays(m, k, n1, n2) and _tower_launches(apart)[0] >= 2, "%d rows" % m
        h = x.astype(np.float64)
        for w, b, a in zip(ws[:2], bs, acts):
            h = _tower_act(h @ w.astype(np.float64) + b, a).astype(np.float16).astype(np.float64)
        z = h @ ws[2].astype(np.float64) + bs[2]
        e = np.exp(z - z.max(1, keepdims=True)) if heads > 1 else z
        want = e / e.sum(1, keepdims=True) if heads > 1 else _sigmoid(z)
        # a hidden value between two fp16s may be rounded to either, 2^-10 of itself apart: of sqrt(sum of squares) about 1 at the next
        # layer, and the result, at most 1 with a slope of at most 1/4, is rounded to 2^-11
        for g in got:
            np.testing.assert_allclose(g, want, rtol=0, atol=4 * 2.0**-11, err_msg="%d rows" % m)


def test_tower_adds_up_as_finely_as_two_launches(pb):
    """An output's sums are as many as in the launches that the tower stands for, which shows in how many probabilities are rounded
    to another fp16 than the exact one: 1.02 times those of two launches here, 1.2 times with one sum over all of 896 inputs."""
    k, n1, n2, rows = 896, 512, 256, 2048
    off = {1: 0, 0: 0}
    for seed in range(4):
        rng = np.random.default_rng(seed)
        ws = [(rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float16) for s in ((k, n1), (n1, n2), (n2, 2))]
        ws[2] = (ws[2] * 4).astype(np.float16)
        bs = [(rng.standard_normal(n) * 0.1).astype(np.float16) for n in (n1, n2, 2)]
        acts = [("PRelu", np.full(n, 0.25, np.float16)) for n in (n1, n2)]
        x = rng.standard_normal((rows, k)).astype(np.float16)
        h = x.astype(np.float64)
        for w, b, a in zip(ws[:2], bs, acts):
            h = _tower_act(h @ w.astype(np.float64) + b, a).astype(np.float16).astype(np.float64)
        z = h @ ws[2].astype(np.float64) + bs[2]
        e = np.exp(z - z.max(1, keepdims=True))
        for chain in (1, 0):
            p = _tower(pb, ws, bs, acts, chain, 2)
            p.feed("x", x)
            p.forward()
            assert (_tower_launches(p)[0] == 1) == (chain == 1)
            off[chain] += int((p.output_asnumpy("p").reshape(rows, 2) != (e / e.sum(1, keepdims=True)).astype(np.float16)).sum())
    assert 0 < off[1] <= 1.1 * off[0], off


# both sides of each line of bz::fc_tower_pays, and of what the kernel takes
@pytest.mark.parametrize("k,n1,n2,rows,one", [(1024, 100, 40, 1, True), (768, 256, 72, 1, True), (768, 320, 64, 1199, False), (776, 256, 72, 599, False),
                                              (776, 256, 72, 600, True), (1024, 200, 80, 600, True), (1032, 128, 64, 300, True), (1032, 200, 80, 1200, False),
                                              (1280, 100, 40, 2048, True), (1288, 40, 16, 2048, False), (1024, 512, 256, 1199, False), (1024, 512, 256, 1200, True),
                                              (896, 512, 256, 4096, True), (896, 512, 256, 4097, False), (64, 520, 64, 300, False), (64, 64, 264, 300, False)])
def test_tower_launches(pb, k, n1, n2, rows, one):
    """the launches of a pass as it runs, with nothing timing its operators: one for a tower where that pays, else two or three"""
    ws = [np.full(s, 2.0**-10, np.float16) for s in ((k, n1), (n1, n2), (n2, 2))]
    bs = [np.zeros(n, np.float16) for n in (n1, n2, 2)]
    for chain in (1, 0):
        p = _tower(pb, ws, bs, [("Sigmoid", ), ("Sigmoid", )], chain, 2)
        for m in (rows, 8, rows):
            p.feed("x", np.ones((m, k), np.float16))
            p.forward()
        np.testing.assert_allclose(p.output_asnumpy("p"), 0.5, rtol=1e-3)
        launches, timed = _tower_launches(p)
        assert timed == [0, 0] and (launches == 1) == (one and chain == 1)


@pytest.mark.parametrize("k", [72, 70, 69])
def test_tower_rows_do_not_reach_into_each_other(pb, k):
    """infinities and NaNs in some rows, the last one of a workgroup and of the input among them: the others come out as without"""
    rng = np.random.default_rng(k)
    ws = [(rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float16) for s in ((k, 100), (100, 50), (50, 2))]
    bs = [(rng.standard_normal(n) * 0.1).astype(np.float16) for n in (100, 50, 2)]
    p = _tower(pb, ws, bs, [("PRelu", np.full(100, 0.25, np.float16)), None], 1, 2)
    x = rng.standard_normal((70, k)).astype(np.float16)
    bad = [0, 31, 64, 69]
    got = []
    for values in (None, (np.inf, np.nan, -np.inf, np.inf)):
        y = x.copy()
        if values is not None:
            y[bad, [0, k - 1, k - 1, k - 1]] = values
        p.feed("x", y)
        p.forward()
        got.append(p.output_asnumpy("p").reshape(70, 2).copy())
    rest = [i for i in range(70) if i not in bad]
    np.testing.assert_array_equal(got[0][rest], got[1][rest])
    assert np.isnan(got[1][31]).all()


# k: one input, ragged and whole chunks of four and groups of sixteen, more than one ring of groups a wave, the longest taken; n1, n2: a lane, one
# block of 64 and two, ragged and whole, the most; rows: one to four a workgroup, and the line of bz::fc_rows_pays
@pytest.mark.parametrize("k,n1,n2,heads,rows", [(1, 9, 9, 1, (1, 5)), (4, 64, 63, 2, (3, 128, 129)), (5, 65, 64, 8, (4, 257)), (192, 200, 80, 2, (1, 201, 385)),
                                                (468, 256, 100, 2, (2, 1024, 1025)), (445, 250, 256, 3, (300, 7)), (1280, 130, 40, 1, (130, 514)),
                                                (771, 129, 65, 2, (127, 512))])
@pytest.mark.parametrize("act", ["PRelu", "Dice", "Sigmoid", None])
def test_few_rows_in_one_launch(pb, k, n1, n2, heads, rows, act):
    """fp32 layer -> layer -> skinny layer against 64 bits and against one launch a layer, the rows growing and shrinking past the line
    beyond which it is no launch of its own; and while the operators are timed one by one."""
    rng = np.random.default_rng(k * n1 + n2)
    sizes = (k, n1, n2, heads)
    ws = [(rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float32) for s in zip(sizes, sizes[1:])]
    bs = [(rng.standard_normal(n) * 0.1).astype(np.float32) for n in sizes[1:]]
    acts = []
    for n in (n1, n2):
        p = [rng.uniform(0.1, 0.4, n).astype(np.float32), (rng.standard_normal(n) * 0.1).astype(np.float32), rng.uniform(0.5, 1.5, n).astype(np.float32)]
        acts.append({"PRelu": ("PRelu", p[0]), "Dice": ("Dice", *p), "Sigmoid": ("Sigmoid", ), None: None}[act])
    one, apart = (_tower(pb, ws, bs, acts, chain, heads) for chain in (1, 0))
    for step, m in enumerate(rows + rows[:1]):
        print("few rows %d x %d -> %d -> %d -> %d %s" % (m, k, n1, n2, heads, act), flush=True)
        if step == len(rows):
            one.register_observers(["profile"])
        x = rng.standard_normal((m, k)).astype(np.float32)
        got = []
        for p in (one, apart):
            p.feed("x", x)
            p.forward()
            got.append(p.output_asnumpy("p").astype(np.float64).reshape(m, heads))
        if act is not None and step < len(rows):
            assert (_tower_launches(one)[0] == 1) == (m <= 1024) and _tower_launches(apart)[0] >= 2, "%d rows" % m
        h = x.astype(np.float64)
        for w, b, a in zip(ws[:2], bs, acts):
            h = _tower_act(h @ w.astype(np.float64) + b, a)
        z = h @ ws[2].astype(np.float64) + bs[2]
        e = np.exp(z - z.max(1, keepdims=True)) if heads > 1 else z
        want = e / e.sum(1, keepdims=True) if heads > 1 else _sigmoid(z)
        # a layer's sums, of terms whose squares add up to about 1, are off by at most 0.5 * 2^-24 * sqrt(K / 8) each, three layers' to about
        # 1e-6 together; the result has a slope of at most 1/4
        errors = [np.sqrt(np.mean((g - want)**2)) for g in got]
        for g in got:
            np.testing.assert_allclose(g, want, rtol=0, atol=2e-6, err_msg="%d rows" % m)
        # and no further off than the launches that it stands for, by the mean of many (a single one is off by up to half its last bit, 2^-25,
        # either way; the mean of n such by a part of 1 / sqrt(2 n) more or less)
        if m * heads >= 200:
            assert errors[0] <= 1.1 * errors[1], errors


# both sides of each line of bz::fc_rows_pays, and of what the kernel takes
@pytest.mark.parametrize("k,n1,n2,rows,one", [(192, 200, 80, 1024, True), (192, 200, 80, 1025, False), (732, 256, 100, 1, True), (733, 256, 100, 1, False), (64, 256, 64, 9, True),
                                              (64, 257, 64, 9, False), (1280, 16, 16, 9, True), (1281, 16, 16, 9, False), (64, 64, 256, 9, True), (64, 64, 257, 9, False)])
def test_few_rows_launches(pb, k, n1, n2, rows, one):
    """the launches of a pass as it runs, with nothing timing its operators: one for a tower of few rows where that pays, else two or three"""
    ws = [np.full(s, 2.0**-10, np.float32) for s in ((k, n1), (n1, n2), (n2, 2))]
    bs = [np.zeros(n, np.float32) for n in (n1, n2, 2)]
    for chain in (1, 0):
        p = _tower(pb, ws, bs, [("Sigmoid", ), ("Sigmoid", )], chain, 2)
        for m in (rows, 8, rows):
            p.feed("x", np.ones((m, k), np.float32))
            p.forward()
        np.testing.assert_allclose(p.output_asnumpy("p"), 0.5, rtol=1e-6)
        launches, timed = _tower_launches(p)
        assert timed == [0, 0] and (launches == 1) == (one and chain == 1)


@pytest.mark.parametrize("k", [72, 71, 69])
def test_few_rows_do_not_reach_into_each_other(pb, k):
    """infinities and NaNs in some rows, a workgroup's first and last and the input's last among them: the others come out as without, and an
    infinite sum stays infinite"""
    rng = np.random.default_rng(k)
    ws = [(rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float32) for s in ((k, 100), (100, 50), (50, 2))]
    bs = [(rng.standard_normal(n) * 0.1).astype(np.float32) for n in (100, 50, 2)]
    p = _tower(pb, ws, bs, [("Sigmoid", ), ("Sigmoid", )], 1, 2)
    x = rng.standard_normal((390, k)).astype(np.float32)
    bad, last = [0, 2, 200, 389], [0, k - 1, k - 1, k - 1]
    got = []
    for values in (None, (np.inf, np.nan, -np.inf, np.inf)):
        y = x.copy()
        if values is not None:
            y[bad, last] = values
        p.feed("x", y)
        p.forward()
        got.append(p.output_asnumpy("p").reshape(390, 2).copy())
    rest = [i for i in range(390) if i not in bad]
    np.testing.assert_array_equal(got[0][rest], got[1][rest])
    assert np.isnan(got[1][2]).all()
    for i, c, sign in ((0, 0, 1), (200, k - 1, -1), (389, k - 1, 1)):  # Sigmoid(e^x / (1 + e^x)) of +inf is NaN, of -inf 0: NaN where any output is +inf
        assert np.isnan(got[1][i]).all() == (sign * ws[0][c] > 0).any(), i
