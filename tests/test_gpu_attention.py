"""GPU parity of the NVFP4 attention forward (head dims up to 128): the HIP kernel, through the C ABI, against the
CPU oracle on the same packed operands, and the whole `attention()` call against an fp32 attention at the
tolerance of the reference's test (test/test_attention_bench.py:19-66,178-191)."""
import math

import pytest
import torch

from conftest import make_input
from oracle import attention_oracle as A
from oracle import nvfp4_oracle as T

pytestmark = pytest.mark.gpu

# The kernel and the oracle evaluate the same contract on the same operands; they differ in the order of the
# fp32 sums and in the last bit of exp2, which now and then moves a probability across an e2m1 rounding
# boundary (a step of at most 1/12 of its block maximum).  Elementwise tolerance for that:
ATOL = RTOL = 2e-2


def ops():
    from ac4k_kernel_amd import ops as o
    return o


def sdpa_fp32(q, k, v, layout):
    q, k, v = (t.float() for t in (q, k, v))
    if layout == "BNHD":
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    s = q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1])
    o = torch.softmax(s, dim=-1) @ v
    return o.transpose(1, 2).contiguous() if layout == "BNHD" else o


CASES = [(1, 256, 1, 128, "BNHD"), (1, 64, 1, 128, "BNHD"), (2, 100, 3, 128, "BHND"), (1, 33, 2, 128, "BNHD"),
         (1, 300, 1, 128, "BNHD"), (1, 129, 2, 128, "BHND"), (2, 1, 1, 128, "BNHD"), (1, 1000, 4, 128, "BNHD"),
         # enough (query block, head) pairs that the kernel takes 256 query rows per workgroup, ragged last block
         (1, 300, 200, 128, "BHND"), (2, 513, 100, 128, "BNHD"),
         # head dims below 128: 64 (one 64-chunk), 100 and 40 (the quantizer pads the packed rows to 128 / 64)
         (1, 200, 2, 64, "BNHD"), (2, 150, 3, 100, "BHND"), (1, 77, 2, 40, "BNHD")]


@pytest.mark.parametrize("B,N,H,D,layout", CASES)
def test_attention_against_oracle_and_fp32(B, N, H, D, layout):
    shape = (B, N, H, D) if layout == "BNHD" else (B, H, N, D)
    q, k, v = (make_input(shape, seed=s + N) for s in (1, 2, 3))
    o = ops().attention(q.cuda(), k.cuda(), v.cuda(), layout=layout, precision="nvfp4")
    assert o.shape == shape and o.dtype == torch.bfloat16
    # (1) the oracle on the same inputs (its quantizers are bit-identical to the GPU's, so the operands are too)
    ref = A.attention_nvfp4(q, k, v, layout)
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)
    # (2) fp32 attention at the reference test's tolerance (a single kv position returns the quantized V row
    # itself: nothing averages its rounding, so that case is checked against the oracle only)
    if N < 32:
        return
    full = sdpa_fp32(q, k, v, layout)
    cos = torch.nn.functional.cosine_similarity(o.cpu().float().flatten(), full.flatten(), dim=0).item()
    assert cos > 0.98, cos
    err = (o.cpu().float() - full).abs()
    inside = (err <= 2e-1 + 1e-1 * full.abs()).float().mean().item()
    assert inside > 0.999 and err.max().item() < 0.4, (inside, err.max().item())
    if (B, N, H, D, layout) in CASES[:2]:  # the reference's own cases at its own tolerance
        torch.testing.assert_close(o.cpu().float(), full, atol=2e-1, rtol=1e-1)


def test_mha_entry_point_on_given_operands_and_out_argument():
    """mha_nvfp4_fwd called like the reference calls it (python/ac4k_kernel/ops/attention.py:118-131): operands
    from three quantize calls, the output a permuted view of a BNHD tensor, different query and kv lengths."""
    B, Nq, Nkv, H, D = 2, 70, 190, 2, 128
    q = make_input((B, Nq, H, D), seed=31)
    k, v = make_input((B, Nkv, H, D), seed=32), make_input((B, Nkv, H, D), seed=33)
    o = ops()
    qq, kq, vq = o.quantize(q.cuda(), 1, 3), o.quantize(k.cuda(), 1, 3), o.quantize(v.cuda(), 3, 1, swizzle=True)
    out = torch.full((B, Nq, H, D), 7.0, dtype=torch.bfloat16, device="cuda")
    o.mha_nvfp4_fwd(out.permute(0, 2, 1, 3), *qq, *kq, *vq, 0.05)
    cpu = lambda t3: (t3[0].cpu(), t3[1].cpu().view(torch.uint8), t3[2].cpu())  # noqa: E731
    ref = A.mha_nvfp4_fwd(*cpu(qq), *cpu(kq), *cpu(vq), 0.05)                   # [B,H,Nq,D]
    torch.testing.assert_close(out.permute(0, 2, 1, 3).cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)
    # the quantized operands are the oracle's, bit for bit
    eq = T.quantize_nvfp4(v, 3, 1, True)
    assert torch.equal(vq[0].cpu(), eq[0]) and torch.equal(vq[1].cpu().view(torch.uint8), eq[1])


# Launches whose last round is cut into workgroups of 256, 128 and 64 query rows (one round; 256 blocks and a rest of 4 and
# 124), one kv tile, partial last tiles and groups of waves without a row of their own.
@pytest.mark.parametrize("H,Nq,Nkv,D", [(1, 50, 20, 64), (2, 300, 129, 128), (3, 129, 1030, 128), (40, 513, 256, 64),
                                        (130, 300, 200, 64), (190, 260, 300, 64),
                                        # more than a round of blocks, most of whose rows do not exist: all of them cut in four or in two
                                        (300, 49, 49, 64), (300, 40, 600, 40), (512, 100, 300, 64), (24, 2637, 1100, 64),
                                        # one and two kv tiles in workgroups of 256 and 128 rows and with a cut rest
                                        (256, 200, 128, 64), (512, 100, 77, 128), (260, 256, 100, 64), (256, 256, 256, 64),
                                        (512, 100, 190, 40), (300, 256, 129, 64)])
def test_split_plans(H, Nq, Nkv, D):
    q, k, v = make_input((1, H, Nq, D), seed=41), make_input((1, H, Nkv, D), seed=42), make_input((1, H, Nkv, D), seed=43)
    o = ops().attention(q.cuda(), k.cuda(), v.cuda(), layout="BHND", precision="nvfp4")
    ref = A.attention_nvfp4(q, k, v, "BHND")
    # a p next to the boundary of 4 and 6 in e2m1 goes either way, a third of the largest p of its block: with 77 keys (largest
    # p up to 0.08 of the row sum) 0.027 |v|.  In 6.5 million outputs one row holds such a p, whichever way the rows are cut.
    atol = 0.08 if Nkv == 77 else ATOL
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=atol, rtol=RTOL)


# Row maxima of 2^20 to 2^21 (in log2 units), where the exponent of the largest p of a row may exceed zero by half an ulp of
# the maximum, 1/16: p up to 2^(1/16), a block scale beyond 448.  Workgroups of 256, 128 and 64 query rows.
LARGE = [(256, 256), (128, 256), (3, 300)]


@pytest.mark.parametrize("H,N", LARGE)
def test_large_scores(H, N):
    """Every query is its own nearest key by far, so a row of O is that row of V as the quantizers leave it, times
    Phat / l: l = p is within 2^(+-1/16) of 1 (4.5 %), Phat the e4m3 value next to it, half a step of 32 off 416 (3.9 %)."""
    q, v = make_input((1, H, N, 128), seed=51, std=280.0), make_input((1, H, N, 128), seed=52)
    o = ops().attention(q.cuda(), q.cuda(), v.cuda(), layout="BHND", precision="nvfp4").cpu().float()
    assert torch.isfinite(o).all()
    torch.testing.assert_close(o, A.attention_nvfp4(q, q, v, "BHND").float(), atol=ATOL, rtol=0.045 + 0.039 + 2 ** -8)


@pytest.mark.parametrize("H,N", LARGE[:2])  # whole kv tiles: a position without a key has score 0, which would be the maximum
def test_large_negative_scores(H, N):
    """All keys pushed down by one channel: maxima of -1.43 * 2^20, where an ulp is 1/8.  Eight accumulation steps of S and the
    exponent round, half an ulp each at most, so a p is off by up to 2^(9/16) = 1.48, each p of a row by another factor; the
    2-norm of what that leaves in a weighted mean is below 0.48 of it."""
    q, k, v = (make_input((1, H, N, 128), seed=s) for s in (53, 54, 55))
    q[..., 0], k[..., 0] = 3424.0, -3424.0
    o = ops().attention(q.cuda(), k.cuda(), v.cuda(), layout="BHND", precision="nvfp4").cpu().float()
    assert torch.isfinite(o).all()
    ref = A.attention_nvfp4(q, k, v, "BHND").float()
    assert ((o - ref).norm() / ref.norm()).item() < 0.48


@pytest.mark.parametrize("B,Nq,Nkv,H,D,layout", [(1, 1, 1, 1, 8, "BNHD"), (3, 33, 31, 7, 71, "BNHD"), (2, 65, 257, 12, 64, "BNHD"),
                                                 (2, 65, 257, 12, 64, "BHND"), (1, 64, 33, 5, 127, "BHND"), (1, 200, 2100, 9, 128, "BNHD"),
                                                 (11, 100, 77, 12, 65, "BNHD"), (2, 64, 9000, 3, 100, "BHND"), (1, 40, 48, 2, 7, "BNHD")])
def test_whole_call_equals_operator_by_operator(B, Nq, Nkv, H, D, layout, monkeypatch):
    """The two-launch quantizers of attention() give the operands of the separate ones, so the outputs are equal."""
    from ac4k_kernel_amd import _rocm_ops
    shape = lambda n: (B, n, H, D) if layout == "BNHD" else (B, H, n, D)  # noqa: E731
    q, k, v = (make_input(shape(n), seed=s, outliers=True).cuda() for s, n in ((1, Nq), (2, Nkv), (3, Nkv)))
    got = ops().attention(q, k, v, layout=layout, precision="nvfp4")
    monkeypatch.setattr(_rocm_ops, "attention_nvfp4", lambda *a: False)
    assert torch.equal(got, ops().attention(q, k, v, layout=layout, precision="nvfp4"))


@pytest.mark.parametrize("H,N", LARGE)
def test_negative_scale(H, N):
    """A negative product of the scales goes into Q; workgroups of 256, 128 and 64 query rows."""
    q, k, v = (make_input((1, H, N, 128), seed=s).cuda() for s in (56, 57, 58))
    o = ops()
    qq, kq, vq = o.quantize(q, 2, 3), o.quantize(k, 2, 3), o.quantize(v, 3, 2, swizzle=True)
    out = torch.empty((1, H, N, 128), dtype=torch.bfloat16, device="cuda")
    o.mha_nvfp4_fwd(out, *qq, *kq, *vq, -0.088)
    cpu = lambda t3: (t3[0].cpu(), t3[1].cpu().view(torch.uint8), t3[2].cpu())  # noqa: E731
    ref = A.mha_nvfp4_fwd(*cpu(qq), *cpu(kq), *cpu(vq), -0.088)
    torch.testing.assert_close(out.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


def test_whole_call_on_infinite_and_nan_operands(monkeypatch):
    """Through one C call the same as operator by operator: NaN where that gives NaN, the same values elsewhere."""
    from ac4k_kernel_amd import _rocm_ops
    base = [make_input((1, 3, 150, 64), seed=s).cuda() for s in (1, 2, 3)]
    cases = [(t, x) for t in range(3) for x in (float("inf"), -float("inf"), float("nan"))]
    got = []
    for whole in (True, False):
        if not whole:
            monkeypatch.setattr(_rocm_ops, "attention_nvfp4", lambda *a: False)
        for n, (t, x) in enumerate(cases):
            qkv = [b.clone() for b in base]
            qkv[t][0, 1, 77, 5] = x
            o = ops().attention(*qkv, layout="BHND", precision="nvfp4")
            if whole:
                got.append(o)
            else:
                assert torch.allclose(o, got[n], rtol=0, atol=0, equal_nan=True), (t, x)


@pytest.mark.parametrize("precision", ["nvfp4", "int8+fp8e4m3"])
def test_head_dims_below_eight_go_operator_by_operator(precision):
    from ac4k_kernel_amd import _lib
    q, k, v = (make_input((1, 40, 2, 7), seed=s) for s in (1, 2, 3))
    lib = _lib.load()
    f = lib.ac4k_attention_nvfp4_workspace_bytes if precision == "nvfp4" else lib.ac4k_attention_int8_x_fp8_workspace_bytes
    assert f(1, 2, 40, 40, 7, 7) == -1
    o = ops().attention(q.cuda(), k.cuda(), v.cuda(), layout="BNHD", precision=precision)
    ref = A.attention_nvfp4(q, k, v) if precision == "nvfp4" else A.attention_int8_x_fp8(q, k, v)
    torch.testing.assert_close(o.cpu().float(), ref.float(), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("layout", ["BNHD", "BHND"])
@pytest.mark.parametrize("Dqk,Dv", [(128, 64), (64, 128), (40, 100), (100, 8)])
def test_whole_call_with_another_head_dim_of_v(Dqk, Dv, layout, monkeypatch):
    from ac4k_kernel_amd import _rocm_ops
    shape = lambda n, d: (2, n, 5, d) if layout == "BNHD" else (2, 5, n, d)  # noqa: E731
    q, k, v = make_input(shape(70, Dqk), seed=1).cuda(), make_input(shape(200, Dqk), seed=2).cuda(), make_input(shape(200, Dv), seed=3).cuda()
    got = ops().attention(q, k, v, layout=layout, precision="nvfp4")
    monkeypatch.setattr(_rocm_ops, "attention_nvfp4", lambda *a: False)
    assert got.shape == shape(70, Dv) and torch.equal(got, ops().attention(q, k, v, layout=layout, precision="nvfp4"))


def test_more_heads_than_one_launch_carries():
    """2^23 workgroups of 512 threads are 2^32 threads: with so many heads (one query, one key each) both forwards and both
    whole calls still give what they give for a part of the batches."""
    B, H, P = 4096, 2049, 512
    o = ops()
    g = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda shape, hi, dt: torch.empty(shape, dtype=torch.uint8, device="cuda").random_(1, hi, generator=g).view(dt)  # noqa: E731
    q, k, v = rand((B, H, 1, 16), 127, torch.int8), rand((B, H, 1, 16), 127, torch.int8), rand((B, H, 16, 16), 0x78, torch.float8_e4m3fn)
    one, v_sf = torch.full((B, H, 1), 0.01, device="cuda"), torch.ones((B, H, 16), device="cuda")
    out, part = (torch.empty((n, H, 1, 16), dtype=torch.bfloat16, device="cuda") for n in (B, P))
    o.mha_int8_x_fp8_fwd(out, q, one, 64, k, one, 128, v, v_sf, 0.25)
    for b in range(0, B, P):
        s = slice(b, b + P)
        o.mha_int8_x_fp8_fwd(part, q[s], one[s], 64, k[s], one[s], 128, v[s], v_sf[s], 0.25)
        assert torch.equal(out[s], part)
    del q, k, v, v_sf, one
    q, v = rand((B, H, 1, 32), 255, torch.uint8), rand((B, H, 16, 32), 255, torch.uint8)
    sf, gs = rand((B, H, 1, 16, 4), 0x40, torch.float8_e4m3fn), torch.tensor(0.01, device="cuda")
    out.zero_()
    o.mha_nvfp4_fwd(out, q, sf, gs, q, sf, gs, v, sf, gs, 0.125)
    for b in range(0, B, P):
        s = slice(b, b + P)
        o.mha_nvfp4_fwd(part, q[s], sf[s], gs, q[s], sf[s], gs, v[s], sf[s], gs, 0.125)
        assert torch.equal(out[s], part)
    del q, v, sf
    x = torch.empty((B, H, 1, 16), dtype=torch.bfloat16, device="cuda").normal_(generator=g).clamp_(-4, 4)
    x[x == 0] = 0.5  # (a channel of V without a value is NaN, as the quantizer's contract has it)
    x[::P, 0, 0, 0] = 8.0  # the same global scale for a part
    for precision in ("int8+fp8e4m3", "nvfp4"):
        out = o.attention(x, x, x, layout="BHND", precision=precision)
        for b in range(0, B, P):
            y = x[b:b + P]
            assert torch.equal(out[b:b + P], o.attention(y, y, y, layout="BHND", precision=precision)), precision


def test_attention_argument_checks():
    o = ops()
    q = make_input((1, 16, 1, 128), seed=1).cuda()
    with pytest.raises(AssertionError):
        o.attention(q, q, q, precision="fp16")
    with pytest.raises(AssertionError):
        o.attention(q.float(), q, q)
    q192 = make_input((1, 16, 1, 192), seed=1).cuda()
    for precision in ("nvfp4", "int8+fp8e4m3"):
        with pytest.raises(RuntimeError, match="less than 128"):  # the reference's limit (mha_nvfp4.cu:927-929)
            o.attention(q192, q192, q192, precision=precision)
