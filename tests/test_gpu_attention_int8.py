"""GPU parity of the INT8 (QK) x FP8 (PV) attention forward (head dims up to 128) and of the per-token-block int8
quantizer in front of it: the HIP kernels, through the C ABI, against the CPU oracle on the same operands, and
the whole `attention(..., precision="int8+fp8e4m3")` call against an fp32 attention at the tolerance of the
reference's test (test/test_attention_bench.py:69-177: atol 0.2, rtol 1e-2, cosine similarity > 0.99)."""
import math

import pytest
import torch

from conftest import make_input
from oracle import attention_oracle as A
from oracle import nvfp4_oracle as T

pytestmark = pytest.mark.gpu

# The kernel and the oracle evaluate the same contract on the same operands; they differ in the order of the fp32
# sums and in the last bit of exp2, which now and then moves a probability across an e4m3 rounding boundary.
ATOL = RTOL = 2e-2


def ops():
    from ac4k_kernel_amd import ops as o
    return o


def binding():
    from ac4k_kernel_amd import _rocm_ops
    return _rocm_ops


def sdpa_fp32(q, k, v, layout):
    q, k, v = (t.float() for t in (q, k, v))
    if layout == "BNHD":
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    o = torch.softmax(q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1]), dim=-1) @ v
    return o.transpose(1, 2).contiguous() if layout == "BNHD" else o


@pytest.mark.parametrize("shape,layout,block", [((1, 100, 1, 128), "BNHD", 64), ((2, 3, 333, 128), "BHND", 128),
                                                 ((1, 64, 2, 100), "BNHD", 32), ((2, 2, 17, 12), "BHND", 16),
                                                 ((1, 200, 3, 88), "BNHD", 64)])
def test_token_block_quantizer_bit_exact(shape, layout, block):
    """Scales and int8 values equal the oracle's bit for bit, over ragged last blocks, head dims that are padded
    to 16, both layouts, an all-zero block and an outlier."""
    x = make_input(shape, seed=11, outliers=True)
    if layout == "BHND":
        x[0, 0, :block] = 0  # one block whose scale is 0
    ey, es = A.int8_block_token_quantize(x, layout, block)
    n_dim = 1 if layout == "BNHD" else 2
    import importlib
    front = importlib.import_module("ac4k_kernel_amd.ops.attention")  # the module (`ops.attention` is the function)
    y, s = front._int8_quantize(x.cuda(), layout, n_dim, BLOCK_SIZE=block)
    assert y.dtype == torch.int8 and list(y.shape) == list(ey.shape) and list(s.shape) == list(es.shape)
    assert torch.equal(s.cpu(), es) and torch.equal(y.cpu(), ey)


# the first rows are the reference's own test shapes (test/test_attention_bench.py:69-177), head dims 12 to 128
CASES = [(1, 256, 1, 128, "BNHD"), (1, 100, 1, 128, "BNHD"), (2, 111, 2, 100, "BHND"), (1, 444, 1, 88, "BNHD"),
         (11, 100, 12, 12, "BNHD"), (11, 100, 12, 65, "BNHD"), (2, 330, 3, 100, "BNHD"), (2, 111, 2, 128, "BHND"),
         (1, 129, 2, 128, "BHND"), (2, 1, 1, 128, "BNHD"), (1, 1000, 4, 128, "BNHD"),
         # enough (query block, head) pairs that the kernel takes 256 query rows per workgroup, ragged last block
         (1, 300, 200, 128, "BHND")]


@pytest.mark.parametrize("B,N,H,D,layout", CASES)
def test_attention_against_oracle_and_fp32(B, N, H, D, layout):
    shape = (B, N, H, D) if layout == "BNHD" else (B, H, N, D)
    q, k, v = (make_input(shape, seed=s + N) for s in (1, 2, 3))
    o = ops().attention(q.cuda(), k.cuda(), v.cuda(), layout=layout, precision="int8+fp8e4m3")
    assert o.shape == shape and o.dtype == torch.bfloat16
    ref = A.attention_int8_x_fp8(q, k, v, layout)
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)
    if N < 32:  # a single kv position returns the quantized V row itself: nothing averages its rounding
        return
    full = sdpa_fp32(q, k, v, layout)
    cos = torch.nn.functional.cosine_similarity(o.cpu().float().flatten(), full.flatten(), dim=0).item()
    assert cos > 0.99, cos
    torch.testing.assert_close(o.cpu().float(), full, atol=2e-1, rtol=1e-2)


def test_entry_point_on_given_operands():
    """The C entry point on hand-made operands: different lengths of q and kv, q blocks of 32, scales that are not
    those of a quantizer (a zero scale among them), an output with odd strides; against the oracle."""
    B, H, Nq, Nkv = 2, 3, 77, 200
    g = torch.Generator().manual_seed(5)
    q = torch.randint(-127, 128, (B, H, Nq, 128), generator=g, dtype=torch.int8)
    k = torch.randint(-127, 128, (B, H, Nkv, 128), generator=g, dtype=torch.int8)
    q_sf = torch.rand((B, H, 3), generator=g) * 0.01
    k_sf = torch.rand((B, H, 2), generator=g) * 0.01
    k_sf[0, 0, 1] = 0.0
    v = make_input((B, H, Nkv, 128), seed=6)
    v8, v_sf = T.quantize_fp8(v, 3, 2, 2.25, True)
    ref = A.mha_int8_x_fp8_fwd(q, q_sf, 32, k, k_sf, 128, v8, v_sf, 0.09)
    store = torch.zeros((B, H, Nq, 130), dtype=torch.bfloat16, device="cuda")
    o = store[..., 1:129]
    binding().mha_int8_x_fp8_fwd(o, q.cuda(), q_sf.cuda(), 32, k.cuda(), k_sf.cuda(), 128,
                                 v8.cuda().view(torch.float8_e4m3fn), v_sf.cuda(), 0.09)
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)
    assert (store[..., 0] == 0).all() and (store[..., 129] == 0).all()


@pytest.mark.parametrize("B,Nq,Nkv,H,D,layout", [(1, 1, 1, 1, 8, "BNHD"), (3, 33, 31, 7, 71, "BNHD"), (2, 65, 257, 12, 64, "BNHD"),
                                                 (2, 65, 257, 12, 64, "BHND"), (1, 64, 33, 5, 127, "BHND"), (1, 200, 2100, 9, 128, "BNHD"),
                                                 (11, 100, 77, 12, 65, "BNHD"), (2, 64, 9000, 3, 100, "BHND"), (1, 40, 48, 2, 7, "BNHD"),
                                                 # statistics with one, two, four and eight waves a workgroup (BHND, many heads)
                                                 (80, 20, 49, 8, 40, "BHND"), (80, 20, 100, 8, 64, "BHND"), (100, 9, 127, 6, 128, "BHND"),
                                                 (100, 9, 200, 6, 100, "BHND")])
def test_whole_call_equals_operator_by_operator(B, Nq, Nkv, H, D, layout, monkeypatch):
    """The two-launch quantizers of attention() against the separate operators.  Everything is bit-identical except that
    a channel mean summed in another order may round to the neighbouring bf16 (2^-9 of the mean, far below a step of
    int8): at most a few int8 values of that channel move by one step, 1/127 of the block maximum of one score term."""
    shape = lambda n: (B, n, H, D) if layout == "BNHD" else (B, H, n, D)  # noqa: E731
    q, k, v = make_input(shape(Nq), seed=1), make_input(shape(Nkv), seed=2).float() + 1.5, make_input(shape(Nkv), seed=3)
    q, k, v = q.cuda(), k.to(torch.bfloat16).cuda(), v.cuda()
    got = ops().attention(q, k, v, layout=layout)
    monkeypatch.setattr(binding(), "attention_int8_x_fp8", lambda *a: False)
    want = ops().attention(q, k, v, layout=layout)
    assert (got == want).float().mean().item() > 0.9
    torch.testing.assert_close(got.float(), want.float(), atol=ATOL, rtol=RTOL)
    # one step of int8 in a channel moves a score by |q| max|k| / 127 / sqrt(D), at most 2 % of a p, whatever the size of the outputs
    dims = (1, 3) if layout == "BNHD" else (2, 3)
    assert ((got.float() - want.float()).norm(dim=dims) / want.float().norm(dim=dims)).max().item() < 0.02


def exact_mean_keys(shape, n_dim, seed):
    """Keys whose token mean is 1.5 in every channel and every order of summation: multiples of 1/16, in pairs around it."""
    n = shape[n_dim]
    k = torch.full(shape, 1.5)
    r = (make_input(shape, seed=seed).float().clamp(-4, 4) * 16).round() / 16
    half = r.narrow(n_dim, 0, n // 2)
    k.narrow(n_dim, 0, n // 2).add_(half)
    k.narrow(n_dim, n // 2, n // 2).sub_(half)
    return k.to(torch.bfloat16).cuda()


@pytest.mark.parametrize("B,Nq,Nkv,H,Dqk,Dv,layout", [(1, 1, 1, 1, 8, 8, "BNHD"), (3, 33, 31, 7, 71, 71, "BNHD"), (2, 65, 257, 12, 64, 64, "BHND"),
                                                      (1, 200, 2100, 9, 128, 128, "BNHD"), (2, 64, 9000, 3, 100, 100, "BHND"),
                                                      (80, 20, 49, 8, 40, 40, "BHND"), (2, 70, 200, 5, 128, 64, "BNHD"),
                                                      (2, 70, 200, 5, 64, 128, "BHND"), (2, 70, 200, 5, 40, 100, "BNHD"), (1, 70, 300, 9, 100, 8, "BHND")])
def test_whole_call_with_exact_means_is_bit_identical(B, Nq, Nkv, H, Dqk, Dv, layout, monkeypatch):
    shape = lambda n, d: (B, n, H, d) if layout == "BNHD" else (B, H, n, d)  # noqa: E731
    q, v = make_input(shape(Nq, Dqk), seed=1).cuda(), make_input(shape(Nkv, Dv), seed=3).cuda()
    k = exact_mean_keys(shape(Nkv, Dqk), 1 if layout == "BNHD" else 2, 2)
    got = ops().attention(q, k, v, layout=layout)
    monkeypatch.setattr(binding(), "attention_int8_x_fp8", lambda *a: False)
    want = ops().attention(q, k, v, layout=layout)
    assert torch.equal(got, want) and torch.isfinite(got).all()


# short heads, whose tiles take sums and maxima themselves: edges of spans, of tiles of K (128) and V (256) and of the rule (512 keys, heads)
@pytest.mark.parametrize("B,Nkv,H,Dqk,Dv,layout", [(1, 1, 3, 64, 8, "BNHD"), (2, 32, 4, 128, 64, "BNHD"), (1, 33, 9, 8, 128, "BNHD"), (1, 128, 5, 100, 100, "BNHD"),
                                                   (2, 129, 40, 64, 64, "BNHD"), (1, 255, 12, 40, 96, "BNHD"), (1, 257, 12, 64, 64, "BNHD"),
                                                   (1, 511, 1, 128, 128, "BHND"), (1, 512, 4, 64, 72, "BHND"), (1, 513, 4, 64, 72, "BHND"),
                                                   (2, 300, 40, 64, 64, "BHND"), (64, 49, 32, 32, 32, "BHND"), (64, 49, 33, 32, 32, "BNHD"),
                                                   (128, 65, 32, 72, 128, "BHND")])
def test_short_heads_take_their_own_statistics(B, Nkv, H, Dqk, Dv, layout, monkeypatch):
    shape = lambda n, d: (B, n, H, d) if layout == "BNHD" else (B, H, n, d)  # noqa: E731
    q, v = make_input(shape(21, Dqk), seed=1).cuda(), make_input(shape(Nkv, Dv), seed=3).cuda()
    k = exact_mean_keys(shape(Nkv, Dqk), 1 if layout == "BNHD" else 2, 2)
    for n in (0, Nkv - 1):  # the maximum in the first and in the last token
        w = v.clone()
        w.select(1 if layout == "BNHD" else 2, n).mul_(30.0)
        got = ops().attention(q, k, w, layout=layout)
        with monkeypatch.context() as m:
            m.setattr(binding(), "attention_int8_x_fp8", lambda *a: False)
            want = ops().attention(q, k, w, layout=layout)
        assert torch.equal(got, want) and torch.isfinite(got).all()


# one launch or two, the operands have the same bits: the tiles sum K in the order of the launch that they replace.  Keys whose sums are rounded
# (a mean far from zero, magnitudes over several binades), so that another order shows.  Waves of one class and of several, spans that end early, one span
# and many, heads that are neighbours in memory and not; where the rule takes two launches by itself the shape is there to pin it
@pytest.mark.parametrize("B,Nkv,H,Dqk,Dv,layout,launches", [
    (1, 1, 3, 64, 8, "BNHD", 1), (2, 32, 4, 128, 64, "BNHD", 1), (1, 33, 9, 8, 128, "BNHD", 1), (1, 128, 5, 100, 100, "BNHD", 1),
    (2, 129, 40, 64, 64, "BNHD", 1), (1, 255, 12, 40, 96, "BNHD", 1), (2, 257, 12, 64, 64, "BNHD", 1), (1, 511, 1, 128, 128, "BHND", 1),
    (1, 512, 4, 64, 72, "BHND", 1), (1, 513, 4, 64, 72, "BHND", 2), (2, 300, 40, 64, 64, "BHND", 2), (2, 300, 12, 64, 64, "BHND", 1),
    (64, 49, 32, 32, 32, "BHND", 2), (64, 49, 16, 32, 32, "BNHD", 1), (128, 65, 32, 72, 128, "BHND", 1)])
def test_one_launch_or_two_give_the_same_operands(B, Nkv, H, Dqk, Dv, layout, launches):
    import ctypes
    from ac4k_kernel_amd import _lib
    lib = _lib.load()
    Nq = 70
    shape = lambda n, d: (B, n, H, d) if layout == "BNHD" else (B, H, n, d)  # noqa: E731
    q, k, v = make_input(shape(Nq, Dqk), seed=1), make_input(shape(Nkv, Dqk), seed=2), make_input(shape(Nkv, Dv), seed=3)
    k = ((k.float() + 3.0) * torch.exp2(make_input(k.shape, seed=4).float().mul(3.0).round())).to(torch.bfloat16)
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    bhn = lambda t: (t.stride(0), t.stride(2), t.stride(1)) if layout == "BNHD" else t.stride()[:3]  # noqa: E731
    nbytes = lib.ac4k_attention_int8_x_fp8_workspace_bytes(B, H, Nq, Nkv, Dqk, Dv)
    got = []
    for two in (0, 1):
        ws, ran = torch.zeros((nbytes,), dtype=torch.uint8, device="cuda"), ctypes.c_int(0)
        size = lib.ac4k_debug_attention_quantize_int8_x_fp8(
            q.data_ptr(), *bhn(q), k.data_ptr(), *bhn(k), v.data_ptr(), *bhn(v), B, H, Nq, Nkv, Dqk, Dv, 2.25, ws.data_ptr(), nbytes, two,
            ctypes.byref(ran), torch.cuda.current_stream().cuda_stream)
        assert 0 < size <= nbytes, _lib.load().ac4k_last_error()
        assert ran.value == (2 if two else launches)
        got.append(ws[:size])
    assert torch.equal(*got) and got[0].any()


# numbers of token spans around those that are in flight together, and the most; more channels than lanes of a wave, and few
@pytest.mark.parametrize("spans", [2, 7, 8, 9, 16, 17, 31, 32])
@pytest.mark.parametrize("Dqk,Dv", [(128, 100), (8, 128)])
def test_whole_call_joins_every_span(spans, Dqk, Dv, monkeypatch):
    n = spans * 32 - 5
    q, v = make_input((1, 40, 1, Dqk), seed=1).cuda(), make_input((1, n, 1, Dv), seed=3).cuda()
    k = exact_mean_keys((1, n, 1, Dqk), 1, 2)
    v[0, n - 1] *= 50.0  # the maxima are in the last span
    got = ops().attention(q, k, v)
    monkeypatch.setattr(binding(), "attention_int8_x_fp8", lambda *a: False)
    assert torch.equal(got, ops().attention(q, k, v)) and torch.isfinite(got).all()


@pytest.mark.parametrize("D", [64, 65, 128])
def test_whole_call_takes_views(D):
    """q and k as views of one buffer of q, k and v, k as a view of the other layout, tokens and heads shared by stride 0."""
    B, N, H = 2, 150, 5
    q, v = make_input((B, N, H, D), seed=1).cuda(), make_input((B, N, H, D), seed=3).cuda()
    k = exact_mean_keys((B, N, H, D), 1, 2)
    want = ops().attention(q, k, v)
    calls = []
    whole = binding().attention_int8_x_fp8
    try:
        binding().attention_int8_x_fp8 = lambda *a: calls.append(whole(*a)) or calls[-1]
        fused = torch.stack((q, k, v), dim=2)  # [B, N, 3, H, D]
        assert torch.equal(ops().attention(fused[:, :, 0], fused[:, :, 1], v), want)
        other = k.transpose(1, 2).contiguous().transpose(1, 2)  # the tokens of a head adjacent
        assert torch.equal(ops().attention(q, other, v), want)
        assert torch.equal(ops().attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2).contiguous(), layout="BHND"), want.transpose(1, 2))
        one_q, one_k = q[:, :, :1].expand(B, N, H, D), k[:, :, :1].expand(B, N, H, D)
        assert torch.equal(ops().attention(one_q, one_k, v), ops().attention(one_q.contiguous(), one_k.contiguous(), v))
        assert calls == [True] * 5
    finally:
        binding().attention_int8_x_fp8 = whole


def test_whole_call_on_infinite_and_nan_operands(monkeypatch):
    """Through one C call the same as operator by operator: NaN where that gives NaN, the same values elsewhere."""
    B, N, H, D = 1, 150, 3, 64
    base = [make_input((B, N, H, D), seed=1).cuda(), exact_mean_keys((B, N, H, D), 1, 2), make_input((B, N, H, D), seed=3).cuda()]
    cases = [(t, x) for t in range(3) for x in (float("inf"), -float("inf"), float("nan"), 0.0)]
    got = []
    for whole in (True, False):
        if not whole:
            monkeypatch.setattr(binding(), "attention_int8_x_fp8", lambda *a: False)
        for n, (t, x) in enumerate(cases):
            qkv = [b.clone() for b in base]
            if x == 0.0:
                qkv[t][0, :, 1, 5] = x  # a channel without a value
            else:
                qkv[t][0, 77, 1, 5] = x
            o = ops().attention(*qkv)
            if whole:
                got.append(o)
            else:
                assert torch.allclose(o, got[n], rtol=0, atol=0, equal_nan=True), (t, x)


# Launches whose last round is cut: workgroups of 256, 128 and 64 query rows (one round; 256 of 256 rows and a rest of 4 and
# 124 blocks), one kv tile and partial last tiles, groups without a row of their own; with scales of both signs, which
# turn the order of the scores around.
@pytest.mark.parametrize("H,Nq,Nkv", [(1, 50, 20), (2, 300, 129), (3, 129, 1030), (40, 513, 256), (130, 300, 200), (190, 260, 300),
                                      # more than a round of blocks, most of whose rows do not exist: all of them cut in four or in two
                                      (300, 49, 49), (300, 40, 600), (512, 100, 300), (24, 2637, 1100),
                                      # one and two kv tiles in workgroups of 256 and 128 rows and with a cut rest
                                      (256, 200, 128), (512, 100, 77), (260, 256, 100), (256, 256, 256), (512, 100, 190), (300, 256, 129)])
@pytest.mark.parametrize("signs", [False, True])
def test_split_plans_and_negative_scales(H, Nq, Nkv, signs):
    g = torch.Generator().manual_seed(H + Nq)
    q = torch.randint(-127, 128, (1, H, Nq, 64), generator=g, dtype=torch.int8)
    k = torch.randint(-127, 128, (1, H, Nkv, 64), generator=g, dtype=torch.int8)
    q_sf = (torch.rand((1, H, -(-Nq // 64)), generator=g) + 0.5) * 0.01
    k_sf = (torch.rand((1, H, -(-Nkv // 128)), generator=g) + 0.5) * 0.01
    if signs:
        q_sf *= torch.where(torch.rand(q_sf.shape, generator=g) < 0.5, -1.0, 1.0)
        k_sf *= torch.where(torch.rand(k_sf.shape, generator=g) < 0.5, -1.0, 1.0)
    v8, v_sf = T.quantize_fp8(make_input((1, H, Nkv, 72), seed=6), 3, 2, 2.25, True)
    ref = A.mha_int8_x_fp8_fwd(q, q_sf, 64, k, k_sf, 128, v8, v_sf, 0.125)
    o = torch.zeros((1, H, Nq, 72), dtype=torch.bfloat16, device="cuda")
    binding().mha_int8_x_fp8_fwd(o, q.cuda(), q_sf.cuda(), 64, k.cuda(), k_sf.cuda(), 128,
                                 v8.cuda().view(torch.float8_e4m3fn), v_sf.cuda(), 0.125)
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


# Workgroups of eight waves in whole rounds (no rest, a rest cut in two and in four), cut alike, and of four waves on one, two and more tiles
@pytest.mark.parametrize("H,Nq,Nkv", [(256, 256, 300), (384, 250, 300), (260, 256, 300), (130, 250, 300), (128, 250, 3900), (8, 1100, 700),
                                      (150, 100, 300), (300, 60, 200), (300, 60, 600), (1, 300, 4000)])
@pytest.mark.parametrize("signs", [False, True])
def test_four_and_eight_waves(H, Nq, Nkv, signs):
    test_split_plans_and_negative_scales(H, Nq, Nkv, signs)


# |S| up to 128 * 128 * 128, the largest that the biased sums of the fast loop hold, at ordinary and at denormal products of scales; from
# 2^100 on the loop of the general case takes them (a score apart is then all of the softmax)
@pytest.mark.parametrize("q_log2,k_log2", [(-9, -9), (-70, -70), (55, 44), (60, 44)])
@pytest.mark.parametrize("H,Nq,Nkv", [(1, 40, 500), (256, 256, 300)])
def test_extreme_scores(H, Nq, Nkv, q_log2, k_log2):
    sm_scale = 0.08664339780807495  # times log2(e) 0.125 exactly: every score is a float, and so is its distance from the maximum
    g = torch.Generator().manual_seed(Nq)
    q = torch.randint(0, 2, (1, H, Nq, 1), generator=g).mul(255).sub(128).to(torch.int8).expand(-1, -1, -1, 128).contiguous()
    k = torch.randint(0, 2, (1, H, Nkv, 1), generator=g).mul(255).sub(128).to(torch.int8).expand(-1, -1, -1, 128).contiguous()
    k[:, :, ::3] = torch.randint(-128, 128, k[:, :, ::3].shape, generator=g, dtype=torch.int8)
    q_sf = torch.full((1, H, -(-Nq // 64)), 2.0 ** q_log2)
    k_sf = torch.full((1, H, -(-Nkv // 128)), 2.0 ** k_log2)
    v8, v_sf = T.quantize_fp8(make_input((1, H, Nkv, 64), seed=6), 3, 2, 2.25, True)
    ref = A.mha_int8_x_fp8_fwd(q, q_sf, 64, k, k_sf, 128, v8, v_sf, sm_scale)
    o = torch.zeros((1, H, Nq, 64), dtype=torch.bfloat16, device="cuda")
    binding().mha_int8_x_fp8_fwd(o, q.cuda(), q_sf.cuda(), 64, k.cuda(), k_sf.cuda(), 128,
                                 v8.cuda().view(torch.float8_e4m3fn), v_sf.cuda(), sm_scale)
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


def test_error_behaviour():
    b = binding()
    q = torch.zeros((1, 1, 16, 128), dtype=torch.int8, device="cuda")
    sf = torch.ones((1, 1, 1), device="cuda")
    v = torch.zeros((1, 1, 128, 16), dtype=torch.float8_e4m3fn, device="cuda")
    v_sf = torch.ones((1, 1, 128), device="cuda")
    o = torch.empty((1, 1, 16, 128), dtype=torch.bfloat16, device="cuda")
    b.mha_int8_x_fp8_fwd(o, q, sf, 64, q, sf, 128, v, v_sf, 1.0)
    with pytest.raises(RuntimeError, match="Q must be"):
        b.mha_int8_x_fp8_fwd(o, q.float(), sf, 64, q, sf, 128, v, v_sf, 1.0)
    with pytest.raises(RuntimeError, match="k_quantize_block_size"):
        b.mha_int8_x_fp8_fwd(o, q, sf, 64, q, torch.ones((1, 1, 1), device="cuda"), 64, v, v_sf, 1.0)
    with pytest.raises(RuntimeError, match="multiple of 16"):
        q24 = torch.zeros((1, 1, 16, 24), dtype=torch.int8, device="cuda")
        b.mha_int8_x_fp8_fwd(o, q24, sf, 64, q24, sf, 128, v, v_sf, 1.0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.uint8])
def test_whole_call_takes_bf16_on_one_device_only(dtype):
    """The whole calls hand pointers to kernels that read bf16: everything else is left to the operators, whose checks name it."""
    import importlib
    front = importlib.import_module("ac4k_kernel_amd.ops.attention")
    b, x = binding(), make_input((1, 2, 16, 64), seed=1).cuda()
    for bad in (x.to(dtype), x.cpu()):
        for args in ((bad, x, x), (x, bad, x), (x, x, bad)):
            assert not b.attention_int8_x_fp8(torch.empty_like(x), *args, 2.25, 0.125)
            assert not b.attention_nvfp4(torch.empty_like(x), *args, 0.125)
        assert not b.attention_int8_x_fp8(torch.empty_like(bad), x, x, x, 2.25, 0.125)
    for bad in (x[0], x[:, :1], x[:, :, :8], x[..., :32]):  # other dims, heads, lengths, head dims than the rest
        for o, k, v in ((bad, x, x), (x, bad, x), (x, x, bad)):
            assert not b.attention_int8_x_fp8(o.contiguous(), x, k.contiguous(), v.contiguous(), 2.25, 0.125), (o.shape, k.shape, v.shape)
    y = x.to(dtype)
    for call in (front._int8_x_fp8_attention, front._nvfp4_attention):
        with pytest.raises(RuntimeError):
            call(y, y, y, "BHND")


@pytest.mark.parametrize("precision", ["int8+fp8e4m3", "nvfp4"])
def test_reference_long_sequence_shape(precision):
    """The long shape of the reference's test list, (1, 75600, 1, 128) BNHD (test/test_attention_bench.py:69-77), for
    both precisions, against an fp32 attention evaluated on the GPU in blocks of query rows, at the reference's
    tolerance."""
    B, N, H, D = 1, 75600, 1, 128
    g = torch.Generator(device="cuda").manual_seed(9567)
    q, k, v = (torch.empty((B, N, H, D), dtype=torch.float32, device="cuda").normal_(generator=g).to(torch.bfloat16)
               for _ in range(3))
    o = ops().attention(q, k, v, layout="BNHD", precision=precision)
    kf, vf = k[0, :, 0].float(), v[0, :, 0].float()
    ref = torch.empty((N, D), dtype=torch.float32, device="cuda")
    for m0 in range(0, N, 4096):
        s = (q[0, m0:m0 + 4096, 0].float() @ kf.t()) / math.sqrt(D)
        ref[m0:m0 + 4096] = torch.softmax(s, dim=-1) @ vf
    got = o[0, :, 0].float()
    cos = torch.nn.functional.cosine_similarity(got.flatten(), ref.flatten(), dim=0).item()
    rtol, stol = (1e-2, 0.99) if precision == "int8+fp8e4m3" else (1e-1, 0.98)
    assert cos > stol, cos
    torch.testing.assert_close(got, ref, atol=2e-1, rtol=rtol)


@pytest.mark.parametrize("precision", ["int8+fp8e4m3", "nvfp4"])
def test_random_shapes(precision):
    """Seeded random batch sizes, head counts, lengths around the tile and block boundaries, head dims and layouts,
    some with outliers: the whole `attention()` call against the oracle."""
    import random
    rnd = random.Random(2024 if precision == "nvfp4" else 4202)
    for t in range(14):
        B, H = rnd.choice([1, 1, 2, 3]), rnd.choice([1, 2, 3, 5, 40])
        N = rnd.choice([1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 511, 777])
        if H == 40:
            N = min(N, 300)
        D = rnd.choice([128, 128, 64, 100, 40, 88, 96, 16, 120])
        layout = rnd.choice(["BNHD", "BHND"])
        shape = (B, N, H, D) if layout == "BNHD" else (B, H, N, D)
        q, k, v = (make_input(shape, seed=s * 1000 + t, outliers=rnd.random() < 0.3) for s in (1, 2, 3))
        o = ops().attention(q.cuda(), k.cuda(), v.cuda(), layout=layout, precision=precision)
        ref = A.attention_nvfp4(q, k, v, layout) if precision == "nvfp4" else A.attention_int8_x_fp8(q, k, v, layout)
        torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL, msg=lambda m: f"{shape} {layout}: {m}")
