"""GPU parity of the dense path (bz_fc_fused, bz_fc_pack_weight, bz_gemm_strided_batched, bz_activation).

The oracle is the reference's composition Activation(Gemm(x, W, b)) in fp32 (oracle/blaze_oracle.c) plus an
fp64 product used to scale tolerances: MKL's / MFMA's summation orders differ, so the error bound is taken
relative to sum_k |a||b| (the condition of the dot product), not to the possibly cancelled result.
  fp32 path:       |got - want| <= 1e-5 * (sum|a||b| + |bias|)        (contract: rel 1e-5)
  fp16/bf16 path:  |got - want| <= 2e-3 * (sum|a||b| + |bias|) (+ out rounding)   (contract: 2e-3)
where want is computed from the same fp16/bf16-rounded inputs the kernel reads.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ACT = {"none": 0, "prelu": 1, "dice": 2, "relu": 3, "sigmoid": 4, "softmax": 5}


@pytest.fixture(scope="module")
def bz():
    import torch
    import blaze_hip
    assert torch.cuda.is_available(), "no GPU visible"
    blaze_hip.device_check()
    return blaze_hip


def _dev(x, dtype=None):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    return t if dtype is None else t.to(dtype)


def _tdtype(name):
    import torch
    return {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[name]


def _round_to(x, name):
    """numpy fp32 array rounded to the kernel's input precision (returned as fp32)."""
    import torch
    if name == "f32":
        return x.astype(np.float32)
    return torch.from_numpy(x.astype(np.float32)).to(_tdtype(name)).to(torch.float32).numpy()


def _fc_case(bz, oracle, M, N, K, in_name, out_name, act, seed, trans_b=False, lda_pad=0, full_bias=False, alpha=1.0,
             beta=1.0, bias=True):
    import torch
    rng = np.random.default_rng(seed)
    A = _round_to(rng.standard_normal((M, K)), in_name)
    Wkn = _round_to(rng.standard_normal((K, N)) / np.sqrt(K), in_name)
    b = None
    if bias:
        b = (rng.standard_normal((M, N) if full_bias else N) * 0.1).astype(np.float32)
    params_np, act_kwargs = (), {}
    if act == "prelu":
        params_np = (rng.uniform(0.1, 0.4, N).astype(np.float32),)
    elif act == "dice":
        params_np = ((rng.standard_normal(N) * 0.1).astype(np.float32), (rng.standard_normal(N) * 0.1).astype(np.float32),
                     rng.uniform(0.5, 1.5, N).astype(np.float32))
    # device inputs
    a_dev = torch.zeros((M, K + lda_pad), dtype=_tdtype(in_name), device="cuda")
    a_dev[:, :K] = _dev(A, _tdtype(in_name))
    a_view = a_dev[:, :K]
    w_src = _dev(Wkn.T.copy() if trans_b else Wkn, _tdtype(in_name) if in_name != "f32" else None)
    wp = bz.pack_weight(w_src, trans_b, {"f32": bz.F32, "f16": bz.F16, "bf16": bz.BF16}[in_name])
    out = bz.fc_fused(a_view, wp, K, bias=None if b is None else _dev(b), act=ACT[act],
                      act_params=tuple(_dev(p) for p in params_np),
                      out_dtype={"f32": bz.F32, "f16": bz.F16, "bf16": bz.BF16}[out_name], alpha=alpha, beta=beta,
                      act_alpha=0.0)
    torch.cuda.synchronize()
    got = out.to(torch.float32).cpu().numpy()
    # oracle: pre-activation in fp64 (tolerance scale) and the reference composition in fp32
    pre64 = alpha * (A.astype(np.float64) @ Wkn.astype(np.float64))
    scale = abs(alpha) * (np.abs(A).astype(np.float64) @ np.abs(Wkn).astype(np.float64))
    if b is not None:
        pre64 = pre64 + beta * b
        scale = scale + np.abs(beta * b)
    pre32 = pre64.astype(np.float32)
    if act == "none":
        want = pre32
    elif act == "prelu":
        want = oracle.prelu(pre32, params_np[0])
    elif act == "dice":
        want = oracle.dice(pre32, *params_np)
    elif act == "relu":
        want = oracle.leaky_relu(pre32, 0.0)
    elif act == "sigmoid":
        want = oracle.sigmoid(pre32)
    else:
        want = oracle.softmax(pre32, 1)
    tol = 1e-5 if in_name == "f32" else 2e-3
    out_eps = {"f32": 0.0, "f16": 2.0**-11, "bf16": 2.0**-8}[out_name]
    # activations on this path are 1-Lipschitz up to the Dice gate (|d/dx| <= 1 + |gamma-1|*0.25*|x|/den): bound by 2
    bound = 2.0 * tol * scale + out_eps * np.abs(want) + 1e-7
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    worst = np.unravel_index(np.argmax(err - bound), err.shape)
    assert np.all(err <= bound), "M=%d N=%d K=%d %s->%s act=%s: err %.3e > bound %.3e at %s (got %r want %r)" % (
        M, N, K, in_name, out_name, act, err[worst], bound[worst], worst, got[worst], want[worst])
    return got, want


def test_reference_gemm_kat_on_gpu(bz, kats):
    import torch
    from test_oracle_pins import _tensor
    c = kats["gemm_net_v1_cpu"]
    A, B, bias = (_tensor(c["tensors"][n]) for n in ("A_output", "B_output", "Bias_output"))
    wp = bz.pack_weight(_dev(B), False, bz.F32)
    out = bz.fc_fused(_dev(A), wp, 3, bias=_dev(bias))
    torch.cuda.synchronize()
    np.testing.assert_allclose(out.cpu().numpy(), np.array(c["expected"]["output"]["values"], np.float32).reshape(2, 2),
                               rtol=0, atol=1e-6)


def test_pack_weight_layout_and_rounding(bz):
    import torch
    rng = np.random.default_rng(0)
    W = rng.standard_normal((37, 21)).astype(np.float32)  # [K, N]
    for trans_b in (False, True):
        src = _dev(W.T.copy() if trans_b else W)
        for dt, tdt in ((bz.F32, torch.float32), (bz.F16, torch.float16), (bz.BF16, torch.bfloat16)):
            p = bz.pack_weight(src, trans_b, dt)
            torch.cuda.synchronize()
            assert p.shape == (21, 40)
            want = torch.from_numpy(W.T.copy()).to(tdt)
            assert torch.equal(p[:, :37].cpu(), want)
            assert not p[:, 37:].cpu().to(torch.float32).numpy().any()


@pytest.mark.parametrize("M,N,K", [(128, 200, 192), (128, 80, 200), (1, 80, 200), (33, 70, 20), (257, 129, 162),
                                   (4100, 1000, 72), (4096, 2048, 64)])
@pytest.mark.parametrize("act", ["none", "prelu", "dice", "relu", "sigmoid"])
def test_fc_fp32(bz, oracle, M, N, K, act):
    print("case fp32 M=%d N=%d K=%d act=%s" % (M, N, K, act), flush=True)
    _fc_case(bz, oracle, M, N, K, "f32", "f32", act, seed=M * 7 + N + K)


@pytest.mark.parametrize("in_name,out_name", [("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("M,N,K,act", [(2048, 512, 896, "prelu"), (2048, 256, 512, "prelu"), (300, 80, 216, "dice"),
                                       (300, 40, 80, "dice"), (64, 200, 168, "dice"), (4096, 2048, 256, "relu"),
                                       (4100, 1000, 200, "dice"), (33000, 80, 216, "dice"), (100, 100, 104, "none"),
                                       (4000, 4104, 72, "prelu"),  # 16 x 17 tiles of 256x256, ragged in M and N
                                       # the software-pipelined K loop: 128x256 tiles (128x128 for fp32 output), ragged
                                       # in M and N, K ending inside a tile and the loop padded with absent tiles
                                       (8200, 1000, 520, "prelu"), (33000, 250, 136, "dice")])
def test_fc_half(bz, oracle, in_name, out_name, M, N, K, act):
    print("case %s->%s M=%d N=%d K=%d act=%s" % (in_name, out_name, M, N, K, act), flush=True)
    _fc_case(bz, oracle, M, N, K, in_name, out_name, act, seed=M + N * 3 + K)


# Up to 512 32x32 tiles (2-byte operands 256, or 192 where rows start on no 16 bytes and K is at most 256) go to the
# kernel whose eight waves share K in units of 128 bytes, 2-byte ones of K above 256 up to 512 tiles to the same with four;
# beyond that, rows that start on no 16 bytes go to the staged tiles with loads at any element.
@pytest.mark.parametrize("in_name,out_name", [("f32", "f32"), ("f16", "f16"), ("bf16", "f32")])
@pytest.mark.parametrize("M,N,K,act,kw", [
    (1, 9, 1, "none", {}), (33, 40, 3, "prelu", {}), (31, 64, 31, "dice", {}),   # a partial unit only
    (32, 32, 64, "relu", {}), (65, 33, 65, "dice", {}),                          # whole units and one element
    (7, 100, 2075, "sigmoid", {}), (96, 70, 1023, "prelu", {"full_bias": True}),  # units a wave, ragged; a bias a row
    (40, 24, 513, "none", {"alpha": 0.5, "beta": 2.0}),
    (1024, 512, 77, "dice", {}), (1025, 512, 77, "dice", {}),                     # 512 tiles, and one row of tiles more
    (3000, 200, 5, "relu", {}), (2100, 300, 9, "none", {"full_bias": True}),      # staged: K about a chunk
    (2049, 513, 80, "prelu", {}), (4100, 200, 33, "none", {"full_bias": True}),   # 64x64, fp32: two groups of waves on each K tile
    (3000, 700, 72, "dice", {}), (2100, 1000, 65, "relu", {}), (4100, 500, 136, "sigmoid", {}), (2048, 1000, 72, "none", {}),  # 2-byte: 128x128 and, one round of tiles, 64x128
    (4100, 1000, 73, "prelu", {}), (8200, 1000, 201, "dice", {}), (33000, 80, 215, "dice", {}),  # 64x128, 128x128, 128x96
    (2100, 300, 256 + 5, "prelu", {}), (3000, 200, 255, "dice", {}), (4100, 200, 769, "relu", {}),  # off 16 bytes: K tiles one and two in flight
    (512, 512, 80, "dice", {}), (513, 512, 80, "dice", {}), (1024, 512, 264, "prelu", {}),  # 2-byte: 256 tiles, one row more; two K tiles in flight
    (384, 512, 77, "relu", {}), (385, 512, 77, "relu", {}), (512, 512, 257, "none", {}), (520, 512, 257, "none", {}),  # the same off 16 bytes
    (1000, 500, 600, "dice", {"full_bias": True}), (1024, 512, 1001, "sigmoid", {}), (730, 512, 64, "relu", {}),  # four waves; one K tile
    (1025, 512, 80, "relu", {}), (2049, 513, 520, "dice", {}), (2049, 513, 508, "none", {}), (4097, 512, 520, "prelu", {}),  # fp32: 64x64, shared by eight waves from K 512 and up to 511 tiles
    (2049, 4097, 513, "none", {}),                                # fp32 off 16 bytes: 128x128 once K is deep
])
def test_fc_few_tiles_and_any_row_start(bz, oracle, in_name, out_name, M, N, K, act, kw):
    print("case any %s M=%d N=%d K=%d act=%s %r" % (in_name, M, N, K, act, kw), flush=True)
    _fc_case(bz, oracle, M, N, K, in_name, out_name, act, seed=M + 5 * N + K, **kw)


@pytest.mark.parametrize("in_name", ["f16", "bf16"])
@pytest.mark.parametrize("K", [8, 9, 15, 63, 65, 71, 445, 513])  # a chunk, its remainders, the unit of 64 and one more, more than one unit a wave
def test_fc_split_reads_nothing_of_a_ragged_row_but_its_own(bz, K, in_name):
    """The unit that K ends in is read from in front of its start and shifted: the numbers behind K of a wider row, NaNs here, and those in front
    of it, count in nothing: every output is the same as without them."""
    import torch
    tdt, dt = {"f16": (torch.float16, bz.F16), "bf16": (torch.bfloat16, bz.BF16)}[in_name]
    g = torch.Generator(device="cuda").manual_seed(K)
    M, N = 33, 65
    wide = torch.full((M, K + 11), float("nan"), device="cuda", dtype=tdt)
    wide[:, :K] = torch.randn((M, K), generator=g, device="cuda").to(tdt)
    w = bz.pack_weight(torch.randn((K, N), generator=g, device="cuda") / K**0.5, False, dt)
    w[:, K:] = float("nan")
    bias = torch.randn(N, generator=g, device="cuda")
    outs = []
    for a in (wide[:, :K], wide[:, :K].contiguous()):
        y = torch.zeros((M, N), device="cuda", dtype=tdt)
        bz.fc_fused(a, w, K, bias=bias, out=y, act=bz.ACT_LEAKY_RELU, act_alpha=0.25)
        outs.append(y)
    want = wide[:, :K].double() @ w[:, :K].double().t() + bias.double()
    want = torch.where(want >= 0, want, 0.25 * want)
    assert torch.equal(outs[0], outs[1])
    # (sums of about 1 in fp32, rounded once to 2^-11 or 2^-8 of themselves)
    torch.testing.assert_close(outs[0].double(), want, rtol=2.0**-10 if in_name == "f16" else 2.0**-7, atol=1e-5)


def _fp32_sum_error(n):
    """Error of an output relative to it, the root mean square over outputs, where every partial sum has n products.  The sum
    grows like sqrt(i) and each step rounds it; rounding is evenly spread over half a unit in the last place either way, which is
    0.425 u of the value in the mean over mantissas (u = 2^-24: u / sqrt(3) times the mean of 1 / m^2, 0.541, to the half).
    So u * 0.425 * sqrt(n / 2); adding a few partial sums and the bias rounds some more: 0.8 u^2.  20 % on top: with half as
    many partial sums it is 41 % more."""
    return 1.2 * 2.0**-24 * (0.425**2 * n / 2 + 0.8)**0.5


@pytest.mark.parametrize("M,N,K", [(4096, 512, 192), (10000, 200, 64), (1500, 700, 400), (2048, 512, 500), (2048, 512, 512), (4096, 512, 896),
                                   (3000, 200, 301), (20000, 256, 162)])
def test_fc_fp32_error_against_64_bits(bz, M, N, K):
    """the staged tiles of one block a wave: four partial sums an output"""
    import torch
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device="cuda")
    w = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bz.F32)
    bias = torch.randn(N, device="cuda") * 0.1
    y = bz.fc_fused(x, w, K, bias=bias)
    want = x.double() @ w[:, :K].double().t().contiguous() + bias.double()
    err = float((y.double() - want).norm() / want.norm())
    assert err <= _fp32_sum_error(K / 4), err


@pytest.mark.parametrize("M,N,K,parts", [(2048, 256, 512, 2), (2048, 128, 1024, 4), (2000, 80, 200, 5), (2049, 256, 512, 2), (4096, 128, 512, 4)])
def test_fc_fp32_error_of_a_layer_with_a_head(bz, M, N, K, parts):
    """up to 2048 rows the 32-column blocks of a row share sixteen waves; beyond, two sums of the 256-wide tile, four of the others"""
    import torch
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device="cuda")
    w = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bz.F32)
    w2 = bz.pack_weight(torch.randn(N, 2, device="cuda"), False, bz.F32)
    bias = torch.randn(N, device="cuda") * 0.1
    z = torch.empty((M, 2), device="cuda")
    y, _ = bz.fc_fused(x, w, K, bias=bias, head=dict(w=w2, act=bz.ACT_NONE, out=z))
    want = x.double() @ w[:, :K].double().t().contiguous() + bias.double()
    err = float((y.double() - want).norm() / want.norm())
    assert err <= _fp32_sum_error(K / parts), err


# 32x64 tiles from 257 of 32x32 on (four waves, two sums each), 32x32 of eight waves for few columns and for few tiles
@pytest.mark.parametrize("M,N,K", [(1024, 512, 896), (300, 1024, 2048), (700, 400, 2048), (700, 512, 400), (16384, 32, 1024), (9000, 20, 512), (500, 256, 1024)])
def test_fc_fp32_error_of_eight_sums(bz, M, N, K):
    """Eight sums an output, K / 8 inputs each in steps of sixteen, each step rounded once or a few times: an error that grows with the
    root of K / 8, 0.26 * 2^-24 of it as measured here.  Half as many sums, the next lower number, would be 1.41 times that."""
    import torch
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device="cuda")
    w = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bz.F32)
    y = bz.fc_fused(x, w, K)
    want = x.double() @ w[:, :K].double().t().contiguous()
    err = float((y.double() - want).norm() / want.norm())
    assert err <= 0.26 * 2.0**-24 * (K / 8) ** 0.5 * 1.15, err


@pytest.mark.parametrize("M,N,K", [(300, 256, 64), (700, 512, 200), (12000, 20, 300), (1024, 512, 300), (2200, 200, 300), (1024, 256, 512)])
@pytest.mark.parametrize("nosqrt", [False, True])
def test_fc_fp32_dice_of_small_layers_is_the_activation_kernels(bz, M, N, K, nosqrt):
    """up to 512 tiles of 32x32 Dice is computed with expf and exact divisions: bit for bit what the standalone kernel makes of the layer"""
    import torch
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device="cuda")
    w = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bz.F32)
    bias = torch.randn(N, device="cuda") * 0.1
    params = (torch.rand(N, device="cuda"), torch.randn(N, device="cuda") * 0.1, torch.rand(N, device="cuda") + 0.2)
    assert -(-M // 32) * -(-N // 32) <= 512
    got = bz.fc_fused(x, w, K, bias=bias, act=bz.ACT_DICE, act_params=params, dice_nosqrt=nosqrt)
    want = bz.activation(bz.fc_fused(x, w, K, bias=bias), bz.ACT_DICE, params, dice_nosqrt=nosqrt)
    assert torch.equal(got, want), float((got - want).abs().max())


# up to 512 tiles of 32x32 that make more than 128 of 64x64, their edges being half empty: 64x64 of eight waves
@pytest.mark.parametrize("M,N,K", [(5000, 90, 896), (4097, 65, 512), (5425, 96, 300), (3000, 150, 1024), (2200, 200, 896), (1700, 270, 2048), (1409, 321, 401)])
def test_fc_fp32_error_of_eight_sums_in_ragged_layers(bz, M, N, K):
    """as above"""
    assert -(-M // 32) * -(-N // 32) <= 512 and -(-M // 64) * -(-N // 64) > 128
    test_fc_fp32_error_of_eight_sums(bz, M, N, K)


# 2-byte layers of more than 256 tiles of 64x64: 64x128 and 128x64 tiles, also for rows that start on no 16 bytes
@pytest.mark.parametrize("in_name,out_name", [("f16", "f16"), ("bf16", "f32")])
@pytest.mark.parametrize("M,N,K,act,kw", [(1900, 520, 392, "dice", {}), (6017, 136, 64, "prelu", {"full_bias": True}),   # 64x128, ragged; one K tile
                                          (16449, 64, 136, "relu", {}), (16448, 33, 72, "dice", {}), (17001, 9, 192, "none", {"full_bias": True}),  # 128x64
                                          (16449, 40, 65, "prelu", {}), (2049, 513, 255, "dice", {}), (2050, 520, 9, "none", {}),   # off 16 bytes: one K tile in flight
                                          (16449, 64, 257, "relu", {}), (3000, 390, 301, "sigmoid", {"full_bias": True}), (2049, 520, 523, "prelu", {})])  # two
def test_fc_two_byte_layers_beyond_one_round_of_tiles(bz, oracle, in_name, out_name, M, N, K, act, kw):
    print("case round %s M=%d N=%d K=%d act=%s %r" % (in_name, M, N, K, act, kw), flush=True)
    assert -(-M // 64) * -(-N // 64) > 256
    _fc_case(bz, oracle, M, N, K, in_name, out_name, act, seed=M + N + K, **kw)


def _plain_bound(x, w, bias):
    """what any order of K fp32 products and sums stays within, and a split that drops 2^-24 of a product"""
    return (x.shape[1] + 8) * 2.0**-24 * (x.double().abs() @ w.double().abs().t().contiguous() + bias.double().abs())


@pytest.mark.parametrize("M,N,K", [(1, 9, 4), (31, 33, 5), (33, 65, 15), (32, 32, 16), (65, 31, 17), (3, 300, 127), (130, 90, 2075), (257, 257, 33),
                                   (700, 512, 201), (520, 520, 600), (1000, 500, 257), (2300, 260, 97), (9000, 130, 130), (1100, 500, 600),
                                   (2111, 321, 203), (3000, 700, 1000)])
@pytest.mark.parametrize("off", [0, 1])
def test_fc_fp32_on_bf16_pieces(bz, M, N, K, off):
    """fp32 layers as products of three bf16s a float: edges of tiles, of a stage of 16 and of its chunks, waves without a stage,
    rows that start on no 16 bytes"""
    import torch
    torch.manual_seed(M + 3 * N + K)
    held = torch.randn(M * (K + off) + off, device="cuda")
    x = held[off:].view(M, K + off)[:, :K]
    w = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bz.F32)
    bias = torch.randn(N, device="cuda") * 0.1
    print("case M=%d N=%d K=%d off=%d" % (M, N, K, off), flush=True)
    full = torch.full((M + 1, N + 3), 7.0, device="cuda")
    bz.fc_fused(x, w, K, bias=bias, out=full[:M, :N])
    want = x.double() @ w[:, :K].double().t().contiguous() + bias.double()
    assert ((full[:M, :N].double() - want).abs() <= _plain_bound(x, w[:, :K], bias)).all()
    assert (full[M:] == 7.0).all() and (full[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K", [(40, 70, 130), (1200, 400, 160), (1200, 800, 250)])
def test_fc_fp32_infinities_and_numbers_at_the_ends_of_the_range(bz, M, N, K):
    """numbers that no bf16 is near to, and such whose pieces lie below the smallest bf16"""
    import torch
    torch.manual_seed(K)
    x = torch.randn(M, K, device="cuda")
    w = bz.pack_weight(torch.rand(K, N, device="cuda") + 0.5, False, bz.F32)
    bias = torch.zeros(N, device="cuda")
    x[0, 3] = float("inf")
    x[1, K - 1] = -float("inf")
    x[2, 7] = float("nan")
    x[3] = 1e-3
    x[3, 5] = 3.402e38
    w[2, :K] *= 2.0**-10  # (a column that takes it without overflow)
    x[4] *= 1e-37
    x[5] = 0.0
    x[6] = -0.0
    x[M - 1] *= 1e-30
    print("case M=%d N=%d K=%d" % (M, N, K), flush=True)
    y = bz.fc_fused(x, w, K, bias=bias)
    want = x.double() @ w[:, :K].double().t().contiguous()
    as32 = want.float()
    assert torch.equal(torch.isnan(y), torch.isnan(as32)) and torch.equal(torch.isposinf(y), torch.isposinf(as32))
    assert torch.equal(torch.isneginf(y), torch.isneginf(as32)) and torch.isfinite(y[3, 2])
    fine = torch.isfinite(as32)
    bound = _plain_bound(x, w[:, :K], bias)
    assert ((y.double() - want).abs() <= bound)[fine].all()
    assert (y[5:7] == 0).all()


@pytest.mark.parametrize("M,N,K", [(40, 70, 130), (1200, 400, 160), (1200, 800, 250), (1024, 512, 300), (1409, 321, 301), (3, 9, 1000)])
def test_fc_fp32_small_numbers_times_large_ones(bz, M, N, K):
    """Operands whose last bits no three bf16s hold, or none at all, times such of the other side that the sums are ordinary numbers, or
    small ones that are not 0; whole rows and columns of them, and single ones among zeros.  Ordinary rows beside them, and rows of
    zeros, come out as without."""
    import torch
    torch.manual_seed(K)
    small = torch.tensor([1.0, 1.2e-38, 1e-40, 1e-41, 1.2e-37, 3.3e-36, 1e-33, 1e14, 1e15], device="cuda", dtype=torch.float64)
    large = torch.tensor([1.0, 1e3, 1e15, 1e18, 1e20, 1e10, 1e-39, 1e-36, 2e-38], device="cuda", dtype=torch.float64)
    plain = torch.randn(M, K, device="cuda")
    x = (plain.double() * small[torch.arange(M, device="cuda") % 9, None]).float()
    w = torch.zeros(N, (K + 3) // 4 * 4, device="cuda")
    w[:, :K] = (torch.randn(N, K, device="cuda").double() * large[torch.arange(N, device="cuda") % 9, None]).float()
    if M > 16:
        x[9] = 0.0
        x[9, 3] = 3e-39
        x[10] = 0.0
        w[11] = 0.0
        w[11, 3] = 1e10
        w[12] = 0.0
    bias = torch.zeros(N, device="cuda")
    print("case M=%d N=%d K=%d" % (M, N, K), flush=True)
    y = bz.fc_fused(x, w, K, bias=bias)
    want = x.double() @ w[:, :K].double().t().contiguous()
    bound = _plain_bound(x, w[:, :K], bias) + K * 2.0**-149  # (below 2^-126 numbers are whole multiples of 2^-149)
    assert (want.abs() < 1e38).all() and (want.abs() > 0).sum() > M * N // 2
    off = (y.double() - want).abs() - bound
    assert (off <= 0).all(), (float((off / bound).max()), int(off.argmax()) // N % 9, int(off.argmax()) % N % 9)
    if M > 16:
        assert (y[10] == 0).all() and (y[:, 12] == 0).all()
        # (rows 0, 9, 18 .. and 7, 16 .. beside others of ordinary numbers)
        ordinary = [r for r in range(M) if r % 9 in (0, 7) and r != 9]
        x1 = plain.clone()
        x1[ordinary] = x[ordinary]
        assert torch.equal(bz.fc_fused(x1, w, K, bias=bias)[ordinary], y[ordinary])


@pytest.mark.parametrize("M,N,K", [(40, 70, 130), (700, 512, 201), (1000, 500, 300), (2048, 512, 899), (1409, 321, 301), (33, 9, 4)])
def test_fc_fp32_tiles_of_sums_that_are_computed_again(bz, M, N, K):
    """an infinity, a NaN or the largest float in every row: all sums again, in a time that does not explode (3.4 of a plain call's at
    2048 x 899 -> 512; 30 as a dot product for each sum)"""
    import torch
    torch.manual_seed(K)
    x = torch.rand(M, K, device="cuda") + 0.5
    plain = x.clone()
    w = bz.pack_weight(torch.rand(K, N, device="cuda") / (4 * K), False, bz.F32)
    rows = torch.arange(M, device="cuda")
    x[rows, rows % K] = torch.tensor([float("inf"), float("nan"), -float("inf"), 3.4028235e38, -3.4e38], device="cuda")[rows % 5]
    print("case M=%d N=%d K=%d" % (M, N, K), flush=True)
    bias = torch.zeros(N, device="cuda")
    y = bz.fc_fused(x, w, K, bias=bias)
    want = x.double() @ w[:, :K].double().t().contiguous()
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isposinf(y), torch.isposinf(want)) and torch.equal(torch.isneginf(y), torch.isneginf(want))
    fine = torch.isfinite(want)
    assert fine.any() and ((y.double() - want).abs() <= _plain_bound(x, w[:, :K], bias))[fine].all()

    def us(a):
        times = []
        for _ in range(20):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(5):
                bz.fc_fused(a, w, K, out=y)
            e1.record()
            e1.synchronize()
            times.append(e0.elapsed_time(e1))
        return sorted(times)[5]
    if M >= 2048:
        assert us(x) < 10 * us(plain)


@pytest.mark.parametrize("M,K,N,H,act", [(1, 1024, 48, 1, "none"), (17, 516, 100, 8, "softmax"), (300, 256, 196, 2, "softmax"), (2049, 512, 256, 2, "none"),
                                         (300, 256, 192, 3, "sigmoid"), (2000, 200, 256, 2, "softmax")])
def test_fc_fp32_head_apart_and_in_the_launch(bz, M, K, N, H, act):
    """below and above k * n = 48 K: with memory for the layer's output, without (in the launch: another stream's call, a capture),
    and with the output left out"""
    import torch
    torch.manual_seed(M + N)
    code = dict(none=bz.ACT_NONE, softmax=bz.ACT_SOFTMAX, sigmoid=bz.ACT_SIGMOID)[act]
    x = torch.randn(M, K, device="cuda")
    w = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bz.F32)
    w2 = bz.pack_weight(torch.randn(N, H, device="cuda") / N**0.5, False, bz.F32)
    bias, bias2 = torch.randn(N, device="cuda") * 0.1, torch.randn(H, device="cuda")
    slope = torch.full((N, ), 0.25, device="cuda")
    wide = x.double() @ w[:, :K].double().t().contiguous() + bias.double()
    wide = torch.where(wide > 0, wide, 0.25 * wide)
    want = wide @ w2[:, :N].double().t().contiguous() + bias2.double()
    want = dict(none=lambda v: v, softmax=lambda v: v.softmax(1), sigmoid=torch.sigmoid)[act](want)
    print("case M=%d K=%d N=%d H=%d %s" % (M, K, N, H, act), flush=True)
    assert bz.lib().bz_fc_head_apart(K, N, bz.F32) == (K * N > 48 << 10) and bz.lib().bz_fc_head_apart(K, N, bz.F16) == 0
    # sums of K and of N terms in any order, the second behind values of about 1 and columns of about N**-0.5
    bound = (K + N + 16) * 2.0**-24 * (1 + wide.abs() @ w2[:, :N].double().abs().t().contiguous())

    def call(store, **kw):
        z, y = torch.full((M, H + 1), 9.0, device="cuda"), torch.full((M, N), 9.0, device="cuda")
        got, _ = bz.fc_fused(x, w, K, bias=bias, act=bz.ACT_PRELU, act_params=(slope, ), out=y, store_out=store,
                             head=dict(w=w2, bias=bias2, act=code, out=z[:, :H]), **kw)
        return z, y, got

    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    for store, kw in ((True, {}), (False, {}), (False, dict(stream=other))):
        z, y, got = call(store, **kw)
        torch.cuda.synchronize()
        assert ((z[:, :H].double() - want).abs() <= bound).all() and (z[:, H:] == 9.0).all()
        assert got is y if store else got is None and (y == 9.0).all()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z, _, _ = call(False)
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert ((z[:, :H].double() - want).abs() <= bound).all()


# Large 2-byte layers go to the streaming kernel (256x128 tiles, loader waves, operands straight into LDS) once
# ceil(M/256) * ceil(N/128) >= 200, K is a multiple of 64 and at least 512, and the output takes 16-byte stores.
@pytest.mark.parametrize("in_name", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,act,kw", [
    (7000, 1000, 512, "prelu", {}),                 # ragged in M (88 rows in the last tile) and N (104 columns)
    (8192, 1024, 576, "dice", {}),                  # whole tiles, an odd number of K tiles
    (6500, 1032, 640, "none", {"alpha": 0.5, "beta": 2.0}),
    (6600, 1024, 512, "sigmoid", {"bias": False}),
    (6400, 1024, 1024, "relu", {"full_bias": True}),
    (51300, 128, 512, "prelu", {}),                 # one N tile; 201 M tiles: the XCD bands are uneven
])
def test_fc_streaming_kernel(bz, oracle, in_name, M, N, K, act, kw):
    print("case stream %s M=%d N=%d K=%d act=%s %r" % (in_name, M, N, K, act, kw), flush=True)
    assert -(-M // 256) * -(-N // 128) >= 200 and K % 64 == 0 and K >= 512
    _fc_case(bz, oracle, M, N, K, in_name, in_name, act, seed=M + N + K, **kw)


@pytest.mark.parametrize("in_name", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,K,N,N2,act,hact", [
    (2048, 512, 256, 2, "prelu", "softmax"),   # config 2's last two layers: 32x256 tile
    (300, 200, 80, 2, "dice", "softmax"),      # DIN main tower tail: 32x128 tile, ragged M
    (5000, 80, 40, 1, "dice", "none"),         # DIN attention tail: 32x64 tile
    (17000, 80, 40, 1, "dice", "none"),        # the same with enough rows for the 64x64 tile
    (513, 128, 128, 8, "relu", "sigmoid"),     # widest head
    (100, 64, 16, 3, "none", "softmax"),
    (4096, 96, 256, 2, "relu", "sigmoid"),
    (4097, 96, 256, 2, "relu", "sigmoid"),
    (2048, 104, 256, 2, "dice", "softmax"),    # fp32: the last size of sixteen rows a workgroup, and the first beyond
    (2049, 104, 256, 2, "dice", "softmax"),
    (2049, 200, 80, 1, "prelu", "sigmoid"),
    (17, 8, 224, 5, "none", "none"),           # a part of one unit of K, seven column blocks on sixteen waves, a single row left
    (1, 1104, 72, 1, "prelu", "sigmoid"),      # units shared by five parts, K ending inside one
])
def test_fc_with_skinny_head_in_one_launch(bz, oracle, in_name, M, K, N, N2, act, hact):
    """Layer + skinny head in one launch against the same two layers as two launches.  The one-launch form uses a tile
    that spans the whole row, so its fp32 sums run in another order: the first layer's output agrees to one rounding
    of the tensor type, the head to 1e-5 (fp32) / 2e-3 (the head reads the rounded tile as the second launch reads the
    stored tensor), also when the first layer's output is not stored.  The head against the oracle, computed from
    the first layer's own stored output: 1e-5 (fp32) / 2e-3 relative to the operand magnitudes."""
    import torch
    print("case", in_name, M, K, N, N2, act, hact, flush=True)
    rng = np.random.default_rng(M + 3 * K + N)
    tdt, bt = _tdtype(in_name), {"f32": bz.F32, "f16": bz.F16, "bf16": bz.BF16}[in_name]
    A = _round_to(rng.standard_normal((M, K)), in_name)
    W1 = _round_to(rng.standard_normal((K, N)) / np.sqrt(K), in_name)
    W2 = _round_to(rng.standard_normal((N, N2)) / np.sqrt(N), in_name)
    b1 = (rng.standard_normal(N) * 0.1).astype(np.float32)
    b2 = (rng.standard_normal(N2) * 0.1).astype(np.float32)
    params = ()
    if act == "prelu":
        params = (rng.uniform(0.1, 0.4, N).astype(np.float32), )
    elif act == "dice":
        params = ((rng.standard_normal(N) * 0.1).astype(np.float32), (rng.standard_normal(N) * 0.1).astype(np.float32),
                  rng.uniform(0.5, 1.5, N).astype(np.float32))
    a = _dev(A, tdt)
    w1 = bz.pack_weight(_dev(W1, None if in_name == "f32" else tdt), False, bt)
    w2 = bz.pack_weight(_dev(W2, None if in_name == "f32" else tdt), False, bt)
    kw = dict(bias=_dev(b1), act=ACT[act], act_params=tuple(_dev(p) for p in params), out_dtype=bt)
    y_ref = bz.fc_fused(a, w1, K, **kw)
    z_ref = bz.fc_fused(y_ref, w2, N, bias=_dev(b2), act=ACT[hact], out_dtype=bz.F32)
    z1 = torch.full((M, N2), -7.0, dtype=torch.float32, device="cuda")
    y1, _ = bz.fc_fused(a, w1, K, head=dict(w=w2, bias=_dev(b2), act=ACT[hact], out=z1), **kw)
    z2 = torch.full((M, N2), -7.0, dtype=tdt, device="cuda")
    none, _ = bz.fc_fused(a, w1, K, head=dict(w=w2, bias=_dev(b2), act=ACT[hact], out=z2), store_out=False, **kw)
    torch.cuda.synchronize()
    assert none is None
    ulp = {"f32": 1e-5, "f16": 2.0**-10, "bf16": 2.0**-7}[in_name]
    np.testing.assert_allclose(y1.float().cpu().numpy(), y_ref.float().cpu().numpy(), rtol=ulp, atol=ulp)  # sums of O(1) magnitude: absolute part for cancelled values
    tol = 1e-5 if in_name == "f32" else 2e-3
    np.testing.assert_allclose(z1.cpu().numpy(), z_ref.cpu().numpy(), rtol=tol, atol=tol)
    np.testing.assert_allclose(z2.float().cpu().numpy(), z1.cpu().numpy(), rtol=ulp, atol=1e-6)  # same head, rounded to the type
    # oracle: second layer in fp64 from the first layer's stored (rounded) output
    y = y1.float().cpu().numpy().astype(np.float64)
    pre = (y @ W2.astype(np.float64) + b2).astype(np.float32)
    want = {"none": pre, "sigmoid": oracle.sigmoid(pre), "softmax": oracle.softmax(pre, 1)}[hact]
    scale = np.abs(y) @ np.abs(W2).astype(np.float64) + np.abs(b2)
    assert np.all(np.abs(z1.cpu().numpy() - want) <= 1e-5 * scale + 1e-6)  # fp32 head from the stored tile: fp32 accuracy


@pytest.mark.parametrize("in_name", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,K,N", [(2049, 512, 256), (33, 64, 136), (1000, 200, 80), (16400, 80, 40), (17, 72, 16), (1, 8, 256), (1, 64, 24)])
def test_fc_head_of_two_outputs_equals_the_same_two_of_more(bz, in_name, M, K, N):
    """the code of a head is unrolled for two outputs or for eight: the same sums in the same order, so the same bits"""
    import torch
    torch.manual_seed(M + K + N)
    tdt, bt = _tdtype(in_name), {"f32": bz.F32, "f16": bz.F16, "bf16": bz.BF16}[in_name]
    a = torch.randn(M, K, device="cuda").to(tdt)
    w1 = bz.pack_weight(torch.randn(K, N, device="cuda") / K**0.5, False, bt)
    W2 = torch.randn(N, 8, device="cuda") / N**0.5
    b2 = torch.randn(8, device="cuda")
    got = {}
    for n in (1, 2, 3, 8):
        z = torch.full((M, n), -7.0, device="cuda")
        head = dict(w=bz.pack_weight(W2[:, :n].contiguous(), False, bt), bias=b2[:n].contiguous(), act=bz.ACT_SIGMOID, out=z)
        bz.fc_fused(a, w1, K, out_dtype=bt, store_out=False, head=head)
        got[n] = z.cpu().numpy()
    for n in (1, 2, 3):
        np.testing.assert_array_equal(got[n], got[8][:, :n])
    y = (a.double() @ w1[:, :K].double().t().contiguous()).cpu().numpy()
    z = y @ W2.to(tdt).double().cpu().numpy() + b2.double().cpu().numpy()
    # the rounding of N stored outputs of O(1), times weights of 1 / sqrt(N), times a slope of at most 1 / 4; fp32: of the sums
    tol = 8 * {"f32": 2.0**-20, "f16": 2.0**-11, "bf16": 2.0**-8}[in_name]
    np.testing.assert_allclose(got[8], 1 / (1 + np.exp(-z)), rtol=0, atol=tol)


def test_fc_head_limits_are_refused(bz):
    import torch
    a = torch.zeros((64, 512), dtype=torch.float16, device="cuda")
    w = torch.zeros((512, 512), dtype=torch.float16, device="cuda")
    h = torch.zeros((2, 512), dtype=torch.float16, device="cuda")
    z = torch.zeros((64, 2), dtype=torch.float32, device="cuda")
    with pytest.raises(bz.BlazeHipError, match="n <= 256"):
        bz.fc_fused(a, w, 512, head=dict(w=h, out=z))
    w = torch.zeros((128, 512), dtype=torch.float16, device="cuda")
    h = torch.zeros((9, 128), dtype=torch.float16, device="cuda")
    with pytest.raises(bz.BlazeHipError, match="head of 9 outputs"):
        bz.fc_fused(a, w, 512, head=dict(w=h, out=torch.zeros((64, 9), dtype=torch.float32, device="cuda")))


@pytest.mark.parametrize("in_name", ["f32", "f16", "bf16"])
# lanes a row: 1 (less than a chunk, one), 2 to 64, more chunks than lanes; ragged ends; whole and ragged last workgroups, rows beyond the grid's first pass
@pytest.mark.parametrize("M,N,K,act", [(1, 1, 1, "none"), (257, 2, 3, "softmax"), (33, 2, 7, "prelu"), (300, 2, 9, "dice"), (129, 1, 17, "sigmoid"), (65, 5, 33, "softmax"),
                                       (31, 2, 101, "softmax"), (5, 2, 127, "none"), (9, 8, 250, "dice"), (3, 2, 513, "sigmoid"), (6, 1, 2061, "none"), (33000, 2, 259, "softmax")])
def test_fc_skinny_of_any_depth(bz, oracle, in_name, M, N, K, act):
    _fc_case(bz, oracle, M, N, K, in_name, in_name, act, seed=M + N + K)


@pytest.mark.parametrize("in_name", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("M,N,K,act", [(2048, 2, 256, "softmax"), (128, 2, 80, "softmax"), (5000, 1, 40, "none"),
                                       (8192, 1, 256, "sigmoid"), (7, 8, 1000, "prelu"), (3, 3, 12, "dice")])
def test_fc_skinny(bz, oracle, in_name, M, N, K, act):
    print("case skinny %s M=%d N=%d K=%d act=%s" % (in_name, M, N, K, act), flush=True)
    _fc_case(bz, oracle, M, N, K, in_name, "f32", act, seed=M + N + K)


def test_fc_variants(bz, oracle):
    """transB weights, padded lda, unaligned K with element-wise loads, full [M,N] bias, alpha/beta, no bias."""
    _fc_case(bz, oracle, 70, 90, 64, "f16", "f16", "prelu", seed=1, trans_b=True)
    _fc_case(bz, oracle, 70, 90, 162, "f16", "f32", "dice", seed=2, lda_pad=6)     # lda=168: vector loads + K tail
    _fc_case(bz, oracle, 70, 90, 162, "f16", "f32", "dice", seed=3, lda_pad=0)     # lda=162: element-wise loads
    _fc_case(bz, oracle, 70, 90, 50, "f32", "f32", "none", seed=4, lda_pad=1)      # fp32 unaligned
    _fc_case(bz, oracle, 40, 48, 32, "f32", "f32", "none", seed=5, full_bias=True, alpha=0.5, beta=-2.0)
    _fc_case(bz, oracle, 40, 48, 32, "f16", "f32", "relu", seed=6, bias=False)
    _fc_case(bz, oracle, 40, 5, 32, "f16", "f32", "none", seed=7, full_bias=True, alpha=0.5, beta=-2.0)


def test_fc_argument_errors(bz):
    import torch
    a = torch.zeros((4, 8), dtype=torch.float16, device="cuda")
    w = torch.zeros((16, 8), dtype=torch.float16, device="cuda")
    with pytest.raises(bz.BlazeHipError, match="softmax"):
        bz.fc_fused(a, w, 8, act=ACT["softmax"])
    with pytest.raises(bz.BlazeHipError, match="PRelu"):
        bz.fc_fused(a, w, 8, act=ACT["prelu"], act_params=(torch.zeros(3, device="cuda"),))
    with pytest.raises(bz.BlazeHipError, match="unknown activation"):
        bz.fc_fused(a, w, 8, act=99)


# ------------------------------------------------------------------------------ strided batched / matmul family
def _bgemm(bz, A, B, M, N, K, batch, sa, sb, ta, tb, dtype, C0=None, alpha=1.0, beta=0.0):
    import torch
    a, b = _dev(A, dtype), _dev(B, dtype)
    c = torch.zeros((batch, M, N), dtype=dtype, device="cuda") if C0 is None else _dev(C0, dtype)
    bz.gemm_strided_batched(a, b, c, M, N, K, batch, sa, sb, M * N, ta, tb, alpha, beta)
    torch.cuda.synchronize()
    return c.to(torch.float32).cpu().numpy()


@pytest.mark.parametrize("dtype_name", ["f32", "f16"])
@pytest.mark.parametrize("batch,M,N,K", [(1, 1, 1, 1), (5, 1, 7, 65), (6, 32, 32, 64), (5, 33, 31, 65), (3, 17, 5, 83), (2, 65, 63, 129),
                                         (2, 3, 130, 33), (4, 64, 64, 40)])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_bgemm_tile_edges(bz, dtype_name, batch, M, N, K, ta, tb):
    """edges of the 32- and 64-wide tiles and of the 128-byte pieces of K, operands starting off 16-byte boundaries, C scaled in"""
    import torch
    print("case bgemm %s b=%d %dx%dx%d ta=%d tb=%d" % (dtype_name, batch, M, N, K, ta, tb), flush=True)
    dtype = {"f32": torch.float32, "f16": torch.float16}[dtype_name]
    rng = np.random.default_rng(M * 1000 + N * 10 + K)
    A, B, C0 = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(dtype) for s in
                ((batch, K, M) if ta else (batch, M, K), (batch, N, K) if tb else (batch, K, N), (batch, M, N)))
    a, b, c = (torch.cat([t.new_zeros(1), t.reshape(-1)]).cuda()[1:] for t in (A, B, C0))
    bz.gemm_strided_batched(a, b, c, M, N, K, batch, M * K, K * N, M * N, ta, tb, 0.5, -2.0)
    torch.cuda.synchronize()
    want = 0.5 * np.matmul(A.double().numpy().transpose(0, 2, 1) if ta else A.double().numpy(),
                           B.double().numpy().transpose(0, 2, 1) if tb else B.double().numpy()) - 2.0 * C0.double().numpy()
    got = c.double().cpu().numpy().reshape(batch, M, N)
    tol = 1e-5 if dtype_name == "f32" else 2e-3
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    np.testing.assert_allclose(got, want, rtol=20 * tol, atol=20 * tol)


@pytest.mark.parametrize("name", ["matmul_net_v1_cpu", "fused_parallel_matmul_net_v1_cpu", "fused_parallel_matmul_net_v2_cpu",
                                  "fused_parallel_matmul_net_v3_cpu"])
def test_reference_matmul_kats_on_gpu(bz, kats, name):
    import torch
    from test_oracle_pins import _tensor
    c = kats[name]
    op = c["ops"][0]
    A, B = (_tensor(c["tensors"][n]) for n in op["inputs"])
    ta, tb = bool(op["args"].get("transA", 0)), bool(op["args"].get("transB", 0))
    P = op["args"].get("parallel_num", 1)
    M, K = A.shape[-2:]
    if ta:
        M, K = K, M
    N = B.shape[-2] if tb else B.shape[-1]
    exp = c["expected"]["output"]
    want = np.array(exp["values"], np.float32).reshape(exp["shape"])
    ab, bb = A.shape[0] // P, B.shape[0] // P
    cb = max(ab, bb)
    got = np.zeros((P * cb, M, N), np.float32)
    for p in range(P):  # BatchedBroadcastGemm: one strided-batched call per parallel slice (broadcast.h:340-378)
        Ap, Bp = A[p * ab:(p + 1) * ab], B[p * bb:(p + 1) * bb]
        got[p * cb:(p + 1) * cb] = _bgemm(bz, Ap, Bp, M, N, K, cb, 0 if ab == 1 else M * K, 0 if bb == 1 else K * N, ta, tb,
                                          torch.float32)
    np.testing.assert_allclose(got.reshape(want.shape), want, rtol=0, atol=1e-6)


@pytest.mark.parametrize("name", ["fused_parallel_gemm_net_v%d_cpu" % i for i in range(1, 6)])
def test_reference_fused_parallel_gemm_kats_on_gpu(bz, kats, name):
    """FusedParallelGemm = P FCs sharing the input: strided batched with stride_a = 0 (fused_parallel_gemm_op.h:115-129)
    after the batched bias broadcast-assign."""
    import torch
    from test_oracle_pins import _tensor
    c = kats[name]
    op = c["ops"][0]
    ins = [_tensor(c["tensors"][n]) for n in op["inputs"]]
    A, B = ins[0], ins[1]
    ta, tb = bool(op["args"].get("transA", 0)), bool(op["args"].get("transB", 0))
    P = op["args"]["parallel_num"]
    M, K = (A.shape[1], A.shape[0]) if ta else A.shape
    N = B.shape[0] // P if tb else B.shape[1]
    C0 = np.zeros((P, M, N), np.float32)
    beta = 0.0
    if len(ins) > 2:
        C0[:] = ins[2].reshape(P, 1, N)
        beta = 1.0
    got = _bgemm(bz, A, B, M, N, K, P, 0, K * N, ta, tb, torch.float32, C0=C0, alpha=1.0, beta=beta)
    exp = c["expected"]["output"]
    np.testing.assert_allclose(got.reshape(exp["shape"]), np.array(exp["values"], np.float32).reshape(exp["shape"]), rtol=0,
                               atol=1e-6)


@pytest.mark.parametrize("dtype_name", ["f32", "f16"])
def test_attention_weighted_sum(bz, oracle, dtype_name):
    """DIN batchdot: scores [B,T,1] (transA) x history [B,T,D] -> [B,1,D]; config 3 shape B=1024, T=50, D=54."""
    import torch
    rng = np.random.default_rng(3)
    Bn, T, D = 1024, 50, 54
    w = _round_to(rng.standard_normal((Bn, T, 1)), dtype_name)
    H = _round_to(rng.standard_normal((Bn, T, D)) * 0.1, dtype_name)
    got = _bgemm(bz, w, H, 1, D, T, Bn, T, T * D, True, False, _tdtype(dtype_name))
    want = oracle.matmul_op(w, H, transa=True, transb=False)
    scale = np.einsum("btk,btd->bkd", np.abs(w), np.abs(H))
    tol = 1e-5 if dtype_name == "f32" else 2e-3
    assert np.all(np.abs(got - want) <= tol * scale + 1e-7)


# ------------------------------------------------------------------------------ standalone activations
@pytest.mark.parametrize("name,act", [("prelu_net_v1_cpu", 1), ("dice_net_v1_cpu", 2), ("leaky_relu_net_v1_cpu", 3),
                                      ("sigmoid_net_v1_cpu", 4), ("softmax_net_v1_cpu", 5)])
def test_reference_activation_kats_on_gpu(bz, kats, name, act):
    import torch
    from test_oracle_pins import _tensor
    c = kats[name]
    op = c["ops"][0]
    ins = [_tensor(c["tensors"][n]) for n in op["inputs"]]
    out = bz.activation(_dev(ins[0]), act, params=tuple(_dev(p) for p in ins[1:]), act_alpha=op["args"].get("alpha", 0.0))
    torch.cuda.synchronize()
    exp = c["expected"]["output"]
    np.testing.assert_allclose(out.cpu().numpy(), np.array(exp["values"], np.float32).reshape(exp["shape"]), rtol=0,
                               atol=1e-6)


def test_activation_random_vs_oracle(bz, oracle):
    import torch
    rng = np.random.default_rng(11)
    X = (rng.standard_normal((513, 77)) * 3).astype(np.float32)
    g, mu, var = ((rng.standard_normal(77) * 0.1).astype(np.float32), (rng.standard_normal(77) * 0.1).astype(np.float32),
                  rng.uniform(0.5, 1.5, 77).astype(np.float32))
    slope = rng.uniform(0, 1, 77).astype(np.float32)
    xd = _dev(X)
    cases = [(1, (slope,), oracle.prelu(X, slope), {}), (2, (g, mu, var), oracle.dice(X, g, mu, var), {}),
             (2, (g, mu, var), oracle.dice(X, g, mu, var, True), {"dice_nosqrt": True}),
             (3, (), oracle.leaky_relu(X, 0.1), {"act_alpha": 0.1}), (4, (), oracle.sigmoid(X), {}),
             (5, (), oracle.softmax(X, 1), {})]
    for act, params, want, kw in cases:
        got = bz.activation(xd, act, params=tuple(_dev(p) for p in params), **kw)
        torch.cuda.synchronize()
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("in_name,P,M,K,N,act,full_bias", [
    ("f32", 3, 3, 2, 3, "none", False),        # the shape of the reference's fused_parallel_gemm fixtures
    ("f32", 4, 257, 72, 40, "prelu", False),   # ragged M, slices narrower than a tile
    ("f16", 3, 2048, 128, 96, "prelu", False), # tiles straddle slice boundaries (96 per slice, 64- or 128-wide tiles)
    ("f16", 5, 300, 216, 80, "dice", False),
    ("bf16", 2, 1000, 64, 256, "relu", False),
    ("f16", 2, 129, 40, 18, "none", False),    # slice width not a whole number of 16-byte chunks: element-wise stores
    ("f32", 3, 65, 30, 24, "none", True),      # a full [P*M, N] bias (fused_parallel_gemm_op.h:78-94)
    ("bf16", 8, 6400, 512, 136, "prelu", False),  # the streaming kernel (25 x 9 tiles); slices straddle its 128-wide tiles
    ("f16", 4, 13000, 512, 128, "none", True),    # the streaming kernel with a full bias
])
def test_fc_split_outputs_equal_separate_layers(bz, oracle, in_name, P, M, K, N, act, full_bias):
    """P sibling layers on one input as ONE launch (bz_fc_desc.n_split): weights [P*N, K] stacked, bias and activation
    parameters [P*N], slice p written as its own [M, N] matrix.  Against the oracle's FusedParallelGemm
    (fused_parallel_gemm_op.h:43-133) followed by the activation, and bit-equal to P separate launches."""
    import ctypes as C
    import torch
    rng = np.random.default_rng(P * 1000 + M + K + N)
    tdt = _tdtype(in_name)
    a = _round_to(rng.standard_normal((M, K)).astype(np.float32), in_name)
    w = _round_to((rng.standard_normal((P, N, K)) / np.sqrt(K)).astype(np.float32), in_name)   # slice p: [N, K] (transB form)
    bias = (rng.standard_normal((P, M, N) if full_bias else (P, N)) * 0.1).astype(np.float32)
    slope = rng.uniform(0.1, 0.4, (P, N)).astype(np.float32)
    dice = [(rng.standard_normal((P, N)) * 0.1).astype(np.float32), (rng.standard_normal((P, N)) * 0.1).astype(np.float32),
            rng.uniform(0.5, 1.5, (P, N)).astype(np.float32)]
    d_a, d_w = _dev(a).to(tdt), _dev(w.reshape(P * N, K)).to(tdt)
    ldw = (K + 7) // 8 * 8
    d_wp = torch.zeros((P * N, ldw), dtype=tdt, device="cuda")
    d_wp[:, :K] = d_w
    d_bias = _dev(bias.reshape(-1))
    params = {"none": (), "relu": (), "prelu": (_dev(slope.reshape(-1)), ), "dice": tuple(_dev(x.reshape(-1)) for x in dice)}[act]
    code = {"none": bz.ACT_NONE, "relu": bz.ACT_LEAKY_RELU, "prelu": bz.ACT_PRELU, "dice": bz.ACT_DICE}[act]
    y = torch.full((P, M, N), float("nan"), dtype=tdt, device="cuda")

    def desc(a_t, w_t, n, bias_t, ps, y_t):
        d = bz.FcDesc()
        d.a, d.w, d.y, d.bias = a_t.data_ptr(), w_t.data_ptr(), y_t.data_ptr(), bias_t.data_ptr()
        d.lda, d.ldw, d.ldy = K, ldw, N
        d.m, d.n, d.k = M, n, K
        d.in_dtype = d.out_dtype = bz.bz_dtype(tdt)
        d.bias_rows = M if full_bias else 1
        d.alpha = d.beta = 1.0
        d.act, d.act_alpha = code, 0.0
        for name, p_ in zip(("act_p0", "act_p1", "act_p2"), ps):
            setattr(d, name, p_.data_ptr())
        d.act_size = n if act == "prelu" else 0
        return d

    d = desc(d_a, d_wp, P * N, d_bias, params, y)
    d.n_split, d.y_split_stride = N, M * N
    print("split case %s P=%d M=%d K=%d N=%d act=%s full_bias=%s" % (in_name, P, M, K, N, act, full_bias), flush=True)
    bz.check(bz.lib().bz_fc_fused(C.byref(d), None))
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    # oracle: FusedParallelGemm with B stacked [P*N, K] under transB, then the activation per slice
    want = oracle.fused_parallel_gemm_op(a, w.reshape(P * N, K), bias.reshape(P * M, N) if full_bias else bias.reshape(-1), P, False, True)
    want = want.reshape(P, M, N)
    for p in range(P):
        if act == "prelu":
            want[p] = oracle.prelu(want[p], slope[p])
        elif act == "dice":
            want[p] = oracle.dice(want[p], dice[0][p], dice[1][p], dice[2][p])
        elif act == "relu":
            want[p] = oracle.leaky_relu(want[p], 0.0)
    tol = 1e-5 if in_name == "f32" else 2e-3
    np.testing.assert_allclose(got, want, rtol=tol, atol=tol * max(1.0, float(np.abs(want).max())))
    # P separate launches of the same kernel family: the same sums tile by tile is not guaranteed (tile shapes follow N),
    # so equality is asked at the tolerance of one rounding of the tensor type
    y2 = torch.full((P, M, N), float("nan"), dtype=tdt, device="cuda")
    for p in range(P):
        ps = tuple(x[p * N:(p + 1) * N] for x in params)
        b_p = d_bias[p * M * N:(p + 1) * M * N] if full_bias else d_bias[p * N:(p + 1) * N]
        bz.check(bz.lib().bz_fc_fused(C.byref(desc(d_a, d_wp[p * N:(p + 1) * N], N, b_p, ps, y2[p])), None))
    torch.cuda.synchronize()
    np.testing.assert_allclose(got, y2.float().cpu().numpy(), rtol=tol, atol=tol * max(1.0, float(np.abs(want).max())))


def test_fc_split_argument_errors(bz):
    import ctypes as C
    import torch
    a = torch.zeros((8, 16), dtype=torch.float16, device="cuda")
    w = torch.zeros((32, 16), dtype=torch.float16, device="cuda")
    y = torch.zeros((2, 8, 16), dtype=torch.float16, device="cuda")
    d = bz.FcDesc()
    d.a, d.w, d.y = a.data_ptr(), w.data_ptr(), y.data_ptr()
    d.lda, d.ldw, d.ldy, d.m, d.n, d.k = 16, 16, 16, 8, 32, 16
    d.in_dtype = d.out_dtype = bz.F16
    d.alpha = 1.0
    d.n_split, d.y_split_stride = 12, 128   # 12 does not divide 32
    assert bz.lib().bz_fc_fused(C.byref(d), None) == -22 and b"n_split" in bz.lib().bz_last_error()
    d.n_split = 16
    d.act = bz.ACT_SOFTMAX
    assert bz.lib().bz_fc_fused(C.byref(d), None) != 0


@pytest.mark.parametrize("dtype_name", ["f32", "f16"])
@pytest.mark.parametrize("B,T,Cn", [(1024, 50, 54), (7, 1, 3), (33, 17, 130), (2, 200, 64),
                                    # fewer channels than steps (first pass or tail pass): the lanes past the last
                                    # channel still hold the weights the others read
                                    (64, 50, 16), (64, 50, 24), (19, 70, 8), (19, 40, 70), (5, 130, 1)])
def test_weighted_pool_equals_mul_matmul_reducesum(bz, oracle, dtype_name, B, T, Cn):
    """bz_weighted_pool against the three launches it replaces (Mul, strided-batched GEMM with transA, ReduceSum), bit
    for bit, and against the oracle's fp32 sums of the rounded operands."""
    import ctypes as C
    import torch
    print("weighted pool %s B=%d T=%d C=%d" % (dtype_name, B, T, Cn), flush=True)
    tdt = _tdtype(dtype_name)
    rng = np.random.default_rng(B + T + Cn)
    x = _round_to(rng.standard_normal((B, T, Cn)), dtype_name)
    w = _round_to(rng.standard_normal((B, T, 1)), dtype_name)
    lens = rng.integers(0, T + 1, B)
    mask = (np.arange(T)[None, :] < lens[:, None]).astype(np.float32).reshape(B, T, 1)
    dx, dw, dm = _dev(x).to(tdt), _dev(w).to(tdt), _dev(mask).to(tdt)
    att, tot = bz.weighted_pool(dx, dw, dm)
    # the separate launches
    aw = bz.broadcast_op(bz.EW_MUL, dw, dm)
    c = torch.empty((B, 1, Cn), dtype=tdt, device="cuda")
    bz.gemm_strided_batched(aw, dx, c, 1, Cn, T, B, T, T * Cn, Cn, trans_a=True)
    s = bz.reduce_sum(dx, 1, keepdims=False)
    torch.cuda.synchronize()
    assert torch.equal(att, c.reshape(B, Cn)) and torch.equal(tot, s)
    # without a mask, and each output alone
    att2, none = bz.weighted_pool(dx, dw, None, want_sum=False)
    bz.gemm_strided_batched(dw, dx, c, 1, Cn, T, B, T, T * Cn, Cn, trans_a=True)
    none2, tot2 = bz.weighted_pool(dx)
    torch.cuda.synchronize()
    assert none is None and none2 is None and torch.equal(att2, c.reshape(B, Cn)) and torch.equal(tot2, s)
    # both outputs as column ranges of a wider matrix, with a third piece copied alongside from a pitched source: the
    # Concat that follows the attention tail, written by the same launch; nothing else of the matrix is touched
    n_copy = 7
    wide = torch.full((B, 2 * Cn + n_copy + 5), 3.0, dtype=tdt, device="cuda")
    src = (torch.arange(B * (n_copy + 3), device="cuda").reshape(B, n_copy + 3) % 251).to(tdt)
    bz.weighted_pool(dx, dw, dm, att_out=wide[:, n_copy + Cn + 2:n_copy + 2 * Cn + 2], sum_out=wide[:, n_copy:n_copy + Cn],
                     copy=(src[:, 1:1 + n_copy], wide[:, :n_copy]))
    torch.cuda.synchronize()
    assert torch.equal(wide[:, :n_copy], src[:, 1:1 + n_copy]) and torch.equal(wide[:, n_copy:n_copy + Cn], tot)
    assert torch.equal(wide[:, n_copy + Cn + 2:n_copy + 2 * Cn + 2], att)
    assert bool((wide[:, n_copy + Cn:n_copy + Cn + 2] == 3.0).all()) and bool((wide[:, n_copy + 2 * Cn + 2:] == 3.0).all())
    bad = bz.WeightedPoolDesc()
    bad.x, bad.w, bad.att = dx.data_ptr(), dw.data_ptr(), wide.data_ptr()
    bad.batch, bad.t, bad.c, bad.dtype, bad.ld_att = B, T, Cn, bz.bz_dtype(tdt), Cn - 1
    if Cn > 1:  # (0 means "c")
        assert bz.lib().bz_weighted_pool(C.byref(bad), None) == -22 and b"ld_att" in bz.lib().bz_last_error()
    bad.ld_att, bad.copy_c = 0, 4  # a piece to copy without its pointers
    assert bz.lib().bz_weighted_pool(C.byref(bad), None) == -22 and b"copied piece" in bz.lib().bz_last_error()
    # oracle: fp32 sums in ascending t of the rounded operands
    wm = _round_to(w * mask, dtype_name)
    want_att = np.zeros((B, Cn), np.float32)
    want_sum = np.zeros((B, Cn), np.float32)
    for t in range(T):
        want_att += wm[:, t, :] * x[:, t, :]
        want_sum += x[:, t, :]
    tol = 1e-5 if dtype_name == "f32" else 2e-3
    np.testing.assert_allclose(att.float().cpu().numpy(), want_att, rtol=tol, atol=tol * max(1.0, np.abs(want_att).max()))
    np.testing.assert_allclose(tot.float().cpu().numpy(), want_sum, rtol=tol, atol=tol * max(1.0, np.abs(want_sum).max()))


def _pieces_desc(bz, pieces, r0, r1, tdt):
    return bz.pieces_desc(pieces, r0, r1, bz.bz_dtype(tdt))


@pytest.mark.parametrize("in_name,out_name", [("f16", "f16"), ("bf16", "bf16"), ("f16", "f32")])
@pytest.mark.parametrize("r0,r1,w,N,act", [(1024, 50, 54, 80, "dice"),   # DIN's attention input in front of its first layer
                                           (37, 5, 8, 96, "prelu"),     # 8 columns a lane, ragged last tile, three column blocks
                                           (300, 1, 40, 24, "none"),    # one column block, K = 160
                                           (64, 3, 56, 40, "relu")])    # K = 224, the most the kernel holds
def test_fc_on_pieces_computed_on_the_fly(bz, oracle, in_name, out_name, r0, r1, w, N, act):
    """bz_fc_fused with a_pieces = [q, k, q-k, q*k] (q broadcast over the second row coordinate) against bz_concat_ew
    followed by the stored-matrix layer, and against the oracle fed the concat's rounded values."""
    import ctypes as C
    import torch
    print("fc on pieces %s->%s r0=%d r1=%d w=%d N=%d act=%s" % (in_name, out_name, r0, r1, w, N, act), flush=True)
    tdt, odt = _tdtype(in_name), _tdtype(out_name)
    rng = np.random.default_rng(r0 + r1 + w + N)
    M, K = r0 * r1, 4 * w
    q = _dev(_round_to(rng.standard_normal((r0, 1, w)), in_name)).to(tdt)
    k = _dev(_round_to(rng.standard_normal((r0, r1, w)), in_name)).to(tdt)
    Wkn = _round_to(rng.standard_normal((K, N)) / np.sqrt(K), in_name)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    params_np = ()
    if act == "prelu":
        params_np = (rng.uniform(0.1, 0.4, N).astype(np.float32), )
    elif act == "dice":
        params_np = ((rng.standard_normal(N) * 0.1).astype(np.float32), (rng.standard_normal(N) * 0.1).astype(np.float32),
                     rng.uniform(0.5, 1.5, N).astype(np.float32))
    params = tuple(_dev(x) for x in params_np)
    wp = bz.pack_weight(_dev(Wkn).to(tdt), False, bz.bz_dtype(tdt))
    pieces = [(bz.EW_ASSIGN, q, None), (bz.EW_ASSIGN, k, None), (bz.EW_SUB, q, k), (bz.EW_MUL, q, k)]
    # two launches
    a_full = bz.concat_ew(pieces).reshape(M, K)
    two = bz.fc_fused(a_full, wp, K, bias=_dev(b), act=ACT[act], act_params=params, out_dtype=bz.bz_dtype(odt), act_alpha=0.0)
    # one launch
    pd = _pieces_desc(bz, pieces, r0, r1, tdt)
    one = torch.full((M, N), float("nan"), dtype=odt, device="cuda")
    d = bz.FcDesc()
    d.a_pieces = C.cast(C.pointer(pd), C.c_void_p)
    d.w, d.y, d.bias = wp.data_ptr(), one.data_ptr(), _dev(b).data_ptr()
    bias_dev = _dev(b)
    d.bias = bias_dev.data_ptr()
    d.ldw, d.ldy = wp.stride(0), N
    d.m, d.n, d.k = M, N, K
    d.in_dtype, d.out_dtype = bz.bz_dtype(tdt), bz.bz_dtype(odt)
    d.bias_rows, d.alpha, d.beta = 1, 1.0, 1.0
    d.act, d.act_alpha = ACT[act], 0.0
    for name, p_ in zip(("act_p0", "act_p1", "act_p2"), params):
        setattr(d, name, p_.data_ptr())
    d.act_size = N if act in ("prelu", "dice") else 0
    bz.check(bz.lib().bz_fc_fused(C.byref(d), None))
    torch.cuda.synchronize()
    got, ref = one.float().cpu().numpy(), two.float().cpu().numpy()
    assert not np.isnan(got).any()
    # oracle on the concat's values (each an fp32 operation rounded once to the tensor type)
    A = a_full.float().cpu().numpy()
    pre = (A.astype(np.float64) @ Wkn.astype(np.float64) + b).astype(np.float32)
    scale = np.abs(A).astype(np.float64) @ np.abs(Wkn).astype(np.float64) + np.abs(b)
    want = {"none": lambda x: x, "relu": lambda x: oracle.leaky_relu(x, 0.0), "prelu": lambda x: oracle.prelu(x, params_np[0]),
            "dice": lambda x: oracle.dice(x, *params_np)}[act](pre)
    out_eps = {"f32": 0.0, "f16": 2.0**-11, "bf16": 2.0**-8}[out_name]
    bound = 2.0 * 2e-3 * scale + out_eps * np.abs(want) + 1e-7
    assert np.all(np.abs(got - want) <= bound)
    assert np.all(np.abs(got - ref) <= bound)


def test_fc_on_pieces_limits_are_refused(bz):
    """outside the kernel's model bz_fc_fused answers BZ_ENOTSUP and launches nothing (the caller runs the concat instead)"""
    import ctypes as C
    import torch
    q = torch.zeros((4, 1, 64), dtype=torch.float16, device="cuda")
    k = torch.zeros((4, 3, 64), dtype=torch.float16, device="cuda")
    wp = torch.zeros((16, 256), dtype=torch.float16, device="cuda")
    y = torch.zeros((12, 16), dtype=torch.float16, device="cuda")
    pieces = [(bz.EW_ASSIGN, q, None), (bz.EW_ASSIGN, k, None), (bz.EW_SUB, q, k), (bz.EW_MUL, q, k)]
    pd = _pieces_desc(bz, pieces, 4, 3, torch.float16)
    d = bz.FcDesc()
    d.a_pieces = C.cast(C.pointer(pd), C.c_void_p)
    d.w, d.y, d.ldw, d.ldy, d.m, d.n, d.k = wp.data_ptr(), y.data_ptr(), 256, 16, 12, 16, 256
    d.in_dtype = d.out_dtype = bz.F16
    d.alpha = 1.0
    assert bz.lib().bz_fc_fused(C.byref(d), None) == bz.ENOTSUP and b"a_pieces" in bz.lib().bz_last_error()  # k = 256 > 224
    pd.op[3] = bz.EW_DIV
    pd.width[0] = pd.width[1] = pd.width[2] = pd.width[3] = 40
    d.k, d.ldw = 160, 160
    assert bz.lib().bz_fc_fused(C.byref(d), None) == bz.ENOTSUP  # a piece that divides


@pytest.mark.parametrize("in_name", ["f16", "bf16"])
@pytest.mark.parametrize("r0,r1,w,N,N2,N3,act2,head_act", [
    (1024, 50, 54, 80, 40, 1, "dice", "none"),     # DIN's attention MLP 216 -> 80 -> 40 -> 1
    (37, 5, 24, 96, 64, 2, "prelu", "softmax"),    # widest second layer, a softmax head, ragged last tile
    (300, 3, 40, 24, 16, 0, "relu", "none"),       # no third layer: the second layer's output is stored
])
def test_attention_mlp_as_one_launch(bz, oracle, in_name, r0, r1, w, N, N2, N3, act2, head_act):
    """bz_fc_fused with a_pieces + next (+ head): the layers after the first run in its launch from rows that never leave
    the chip.  Against the separate launches (concat, layer, layer with its head), which round and store what this one
    only rounds."""
    import ctypes as C
    import torch
    print("attention mlp %s r0=%d r1=%d w=%d %d->%d->%d %s %s" % (in_name, r0, r1, w, N, N2, N3, act2, head_act), flush=True)
    tdt = _tdtype(in_name)
    dt = bz.bz_dtype(tdt)
    rng = np.random.default_rng(r0 + w + N + N2)
    M, K = r0 * r1, 4 * w
    q = _dev(_round_to(rng.standard_normal((r0, 1, w)), in_name)).to(tdt)
    k = _dev(_round_to(rng.standard_normal((r0, r1, w)), in_name)).to(tdt)
    W1 = _dev(_round_to(rng.standard_normal((K, N)) / np.sqrt(K), in_name)).to(tdt)
    W2 = _dev(_round_to(rng.standard_normal((N, N2)) / np.sqrt(N), in_name)).to(tdt)
    b1, b2 = _dev((rng.standard_normal(N) * 0.1).astype(np.float32)), _dev((rng.standard_normal(N2) * 0.1).astype(np.float32))
    dice1 = tuple(_dev(x) for x in ((rng.standard_normal(N) * 0.1).astype(np.float32), (rng.standard_normal(N) * 0.1).astype(np.float32),
                                    rng.uniform(0.5, 1.5, N).astype(np.float32)))
    p2 = {"dice": tuple(_dev(x) for x in ((rng.standard_normal(N2) * 0.1).astype(np.float32), (rng.standard_normal(N2) * 0.1).astype(np.float32),
                                          rng.uniform(0.5, 1.5, N2).astype(np.float32))),
          "prelu": (_dev(rng.uniform(0.1, 0.4, N2).astype(np.float32)), ), "relu": ()}[act2]
    wp1, wp2 = bz.pack_weight(W1, False, dt), bz.pack_weight(W2, False, dt)
    head = None
    if N3:
        W3 = _dev(_round_to(rng.standard_normal((N2, N3)) / np.sqrt(N2), in_name)).to(tdt)
        b3 = _dev((rng.standard_normal(N3) * 0.1).astype(np.float32))
        wp3 = bz.pack_weight(W3, False, dt)
    pieces = [(bz.EW_ASSIGN, q, None), (bz.EW_ASSIGN, k, None), (bz.EW_SUB, q, k), (bz.EW_MUL, q, k)]
    # separate launches
    a_full = bz.concat_ew(pieces).reshape(M, K)
    y1 = bz.fc_fused(a_full, wp1, K, bias=b1, act=bz.ACT_DICE, act_params=dice1)
    if N3:
        z_ref = torch.empty((M, N3), dtype=torch.float32, device="cuda")
        bz.fc_fused(y1, wp2, N, bias=b2, act=ACT[act2], act_params=p2, act_alpha=0.0,
                    head=dict(w=wp3, bias=b3, act=ACT[head_act], out=z_ref), store_out=False)
    else:
        y2_ref = bz.fc_fused(y1, wp2, N, bias=b2, act=ACT[act2], act_params=p2, act_alpha=0.0)
    # one launch
    pd = _pieces_desc(bz, pieces, r0, r1, tdt)
    nx = bz.FcNext()
    nx.w, nx.ldw, nx.n, nx.bias = wp2.data_ptr(), wp2.stride(0), N2, b2.data_ptr()
    nx.alpha = nx.beta = 1.0
    nx.act, nx.act_alpha = ACT[act2], 0.0
    for name, p_ in zip(("act_p0", "act_p1", "act_p2"), p2):
        setattr(nx, name, p_.data_ptr())
    nx.act_size = N2 if act2 in ("prelu", "dice") else 0
    d = bz.FcDesc()
    d.a_pieces = C.cast(C.pointer(pd), C.c_void_p)
    d.next = C.cast(C.pointer(nx), C.c_void_p)
    d.w, d.ldw, d.bias = wp1.data_ptr(), wp1.stride(0), b1.data_ptr()
    d.m, d.n, d.k, d.ldy = M, N, K, N
    d.in_dtype = d.out_dtype = dt
    d.bias_rows, d.alpha, d.beta = 1, 1.0, 1.0
    d.act, d.act_size = bz.ACT_DICE, N
    d.act_p0, d.act_p1, d.act_p2 = (t.data_ptr() for t in dice1)
    if N3:
        z = torch.full((M, N3), float("nan"), dtype=torch.float32, device="cuda")
        d.head_w, d.head_ldw, d.head_bias, d.head_y, d.head_ldy = wp3.data_ptr(), wp3.stride(0), b3.data_ptr(), z.data_ptr(), N3
        d.head_n, d.head_act, d.head_out_dtype = N3, ACT[head_act], bz.F32
    else:
        y2 = torch.full((M, N2), float("nan"), dtype=tdt, device="cuda")
        nx.y, nx.ldy = y2.data_ptr(), N2
    bz.check(bz.lib().bz_fc_fused(C.byref(d), None))
    torch.cuda.synchronize()
    got = (z if N3 else y2).float().cpu().numpy()
    ref = (z_ref if N3 else y2_ref).float().cpu().numpy()
    assert not np.isnan(got).any()
    eps = 2.0**-8 if in_name == "bf16" else 2.0**-11
    # three roundings of the tensor type on the way, each amplified by at most the next layer's row sums (weights ~ 1/sqrt(K))
    np.testing.assert_allclose(got, ref, rtol=0, atol=(8 * eps) * max(1.0, float(np.abs(ref).max())) + 2e-3)
    # also with the first layer's own output stored
    y1_one = torch.full((M, N), float("nan"), dtype=tdt, device="cuda")
    d.y = y1_one.data_ptr()
    bz.check(bz.lib().bz_fc_fused(C.byref(d), None))
    torch.cuda.synchronize()
    np.testing.assert_allclose(y1_one.float().cpu().numpy(), y1.float().cpu().numpy(), rtol=0,
                               atol=4 * eps * max(1.0, float(y1.float().abs().max())))
    np.testing.assert_allclose((z if N3 else y2).float().cpu().numpy(), got, rtol=0, atol=0)


@pytest.mark.parametrize("in_name", ["f16", "bf16"])
@pytest.mark.parametrize("N3,head_act", [(1, "sigmoid"), (2, "none"), (3, "sigmoid"), (8, "softmax")])
def test_attention_mlp_with_heads_of_either_unrolling(bz, oracle, in_name, N3, head_act):
    test_attention_mlp_as_one_launch(bz, oracle, in_name, 37, 5, 24, 96, 64, N3, "prelu", head_act)


@pytest.mark.parametrize("in_name", ["f16", "bf16"])
@pytest.mark.parametrize("r0,r1,w,N,N2,N3,act2,head_act", [
    (1, 1, 8, 16, 16, 1, "dice", "none"),          # the narrowest, one row
    (3, 5, 10, 16, 16, 2, "relu", "softmax"),      # one row short of a tile, a chunk of which six are the one before's
    (16, 1, 30, 24, 40, 3, "prelu", "sigmoid"),    # one tile, half a block
    (17, 1, 32, 40, 64, 8, "dice", "softmax"),     # one row over, a whole step
    (5, 13, 34, 80, 40, 1, "relu", "none"),        # two columns into the next step
    (11, 6, 56, 96, 64, 0, "dice", "none"),        # the widest; no third layer
    (7, 50, 40, 45, 17, 0, "prelu", "none"),
    (9, 7, 48, 33, 9, 0, "dice", "none"),
    (2100, 8, 18, 80, 40, 1, "dice", "none"),      # eight waves a workgroup
    (1500, 50, 24, 80, 40, 2, "dice", "softmax"),  # several tiles a wave, the last ones fewer
    (40, 3, 6, 24, 16, 1, "dice", "none"),         # narrower than a chunk: the general form
])
def test_attention_mlp_at_the_edges_of_its_tiles(bz, oracle, in_name, r0, r1, w, N, N2, N3, act2, head_act):
    test_attention_mlp_as_one_launch(bz, oracle, in_name, r0, r1, w, N, N2, N3, act2, head_act)


@pytest.mark.parametrize("in_name", ["f16", "bf16"])
@pytest.mark.parametrize("w,N,N2", [(54, 80, 17), (24, 50, 9), (8, 33, 63)])
def test_attention_mlp_of_odd_columns_equals_the_padded_one(bz, in_name, w, N, N2):
    """a second layer of columns that are no whole number of blocks, with its head: the bits of the same layer with columns of
    zeros up to the next multiple of sixteen (which add zeros to the head's sums)"""
    import ctypes as C
    import torch
    torch.manual_seed(w + N2)
    tdt, dt = _tdtype(in_name), {"f16": bz.F16, "bf16": bz.BF16}[in_name]
    r0, r1, P = 21, 7, (N2 + 15) // 16 * 16
    M, K = r0 * r1, 4 * w
    q, his = torch.randn(r0, w, device="cuda").to(tdt), torch.randn(M, w, device="cuda").to(tdt)
    W1, W2, W3 = torch.randn(K, N, device="cuda") / K**0.5, torch.zeros(N, P, device="cuda"), torch.zeros(P, 2, device="cuda")
    b2, slope = torch.zeros(P, device="cuda"), torch.full((P, ), 0.25, device="cuda")
    W2[:, :N2], W3[:N2], b2[:N2] = torch.randn(N, N2, device="cuda") / N**0.5, torch.randn(N2, 2, device="cuda"), torch.randn(N2, device="cuda")
    wp1 = bz.pack_weight(W1, False, dt)
    got = []
    for n2 in (N2, P):
        wp2, wp3 = bz.pack_weight(W2[:, :n2].contiguous(), False, dt), bz.pack_weight(W3[:n2].contiguous(), False, dt)
        z = torch.full((M, 2), float("nan"), device="cuda")
        d, pd, nx = bz.FcDesc(), bz.ConcatEwDesc(), bz.FcNext()
        pd.dtype, pd.n, pd.r0, pd.r1 = dt, 4, r0, r1
        for i, (op, x, y) in enumerate(((bz.EW_ASSIGN, q, None), (bz.EW_ASSIGN, his, None), (bz.EW_SUB, q, his), (bz.EW_MUL, q, his))):
            pd.op[i], pd.width[i], pd.x[i] = op, w, x.data_ptr()
            pd.x_stride[i][0], pd.x_stride[i][1] = (w, 0) if x is q else (r1 * w, w)
            if y is not None:
                pd.y[i], pd.y_stride[i][0], pd.y_stride[i][1] = y.data_ptr(), r1 * w, w
        nx.w, nx.ldw, nx.n, nx.bias, nx.act, nx.act_size = wp2.data_ptr(), wp2.stride(0), n2, b2.data_ptr(), bz.ACT_PRELU, n2
        nx.act_p0, nx.alpha, nx.beta = slope.data_ptr(), 1.0, 1.0
        d.a_pieces, d.next = C.addressof(pd), C.addressof(nx)
        d.w, d.ldw, d.m, d.n, d.k, d.ldy, d.in_dtype, d.out_dtype, d.alpha = wp1.data_ptr(), wp1.stride(0), M, N, K, N, dt, dt, 1.0
        d.act = bz.ACT_SIGMOID
        d.head_w, d.head_ldw, d.head_y, d.head_ldy, d.head_n, d.head_out_dtype = wp3.data_ptr(), wp3.stride(0), z.data_ptr(), 2, 2, bz.F32
        d.head_act = bz.ACT_NONE
        bz.check(bz.lib().bz_fc_fused(C.byref(d), None))
        torch.cuda.synchronize()
        got.append(z.cpu().numpy())
    assert not np.isnan(got[0]).any()
    np.testing.assert_array_equal(got[0], got[1])
