"""The C-ABI library: loads, exports every function include/ac4k_nvfp4.h declares, reports
attributes, and rejects bad arguments before touching the GPU (no compute calls here)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "ac4k_nvfp4.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ac4k_[a-z0-9_]+)\s*\(", text)))


def test_header_and_loader_agree():
    from ac4k_kernel_amd import _lib
    names = declared_functions()
    assert len(names) >= 18
    assert sorted(_lib.SIGNATURES) == names
    lib = _lib.load()
    for n in names:
        assert hasattr(lib, n), n


def test_attributes():
    import ac4k_kernel_amd as pkg
    assert pkg.get_backend() == "rocm" and pkg.get_arch() == "gfx950"
    assert pkg.get_info() == {"version": "0.1.0", "backend": "rocm", "arch": "gfx950"}
    from ac4k_kernel_amd import ops
    for name in ["quantize", "linear", "quantize_nvfp4", "quantize_fp8", "quantize_int8", "linear_nvfp4"]:
        assert callable(getattr(ops, name))


def test_product_does_not_import_oracle():
    # the shipped package must not reach into oracle/ (it is the checker, not the product)
    pkg = os.path.join(ROOT, "ac4k_kernel_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                src = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in src, os.path.join(dirpath, f)


def test_argument_rejection_without_gpu():
    from ac4k_kernel_amd import _lib
    lib = _lib.load()
    one = ctypes.c_void_p(16)  # never dereferenced: every call below is rejected during validation
    rc = lib.ac4k_quantize_nvfp4(None, one, one, one, 1, 1, 4, 64, 0, 0, 64, 1, 0, None)
    assert rc != 0 and b"null" in lib.ac4k_last_error()
    rc = lib.ac4k_quantize_nvfp4(one, one, one, one, 1, 1, 0, 64, 0, 0, 64, 1, 0, None)
    assert rc != 0 and b"positive" in lib.ac4k_last_error()
    rc = lib.ac4k_linear_nvfp4(one, 0, one, one, one, one, one, one, None, 0, 4, 4, 24, None)
    assert rc != 0 and b"multiple of 16" in lib.ac4k_last_error()
    rc = lib.ac4k_linear_nvfp4(one, 7, one, one, one, one, one, one, None, 0, 4, 4, 64, None)
    assert rc != 0 and b"bfloat16, half or float" in lib.ac4k_last_error()
    # a sliced view (rows of 64 taken out of rows of 128) is not dense: the global scale would be taken
    # over the wrong elements, so the one-call quantizer refuses it; so it does a zero stride on a real dim
    rc = lib.ac4k_quantize_nvfp4_bf16(one, one, one, one, 1, 1, 4, 64, 0, 0, 128, 1, 0, 2688.0, None)
    assert rc != 0 and b"dense" in lib.ac4k_last_error()
    rc = lib.ac4k_quantize_nvfp4_bf16(one, one, one, one, 1, 3, 4, 64, 0, 0, 64, 1, 0, 2688.0, None)
    assert rc != 0 and b"strides must be positive" in lib.ac4k_last_error()
    # tuning values outside the instantiated kernels are refused, zeros are accepted
    assert lib.ac4k_set_linear_tuning(4, 1, 1, 0, 0) != 0 and b"tile plan" in lib.ac4k_last_error()
    assert lib.ac4k_set_linear_tuning(0, 0, 0, 100, 0) != 0 and b"skinny_ks" in lib.ac4k_last_error()
    assert lib.ac4k_set_linear_tuning(0, 0, 0, 0, 4) != 0 and b"decode_kernel" in lib.ac4k_last_error()
    # a rejected call leaves every earlier field alone: here the decode kernel choice is valid, skinny_ks is not,
    # and the plan of a decode-sized shape stays what the library picks on its own
    before = lib.ac4k_linear_nvfp4_skinny_workspace_bytes(4, 4096, 14336)
    assert lib.ac4k_set_linear_tuning(0, 0, 0, 100, 2) != 0
    assert lib.ac4k_linear_nvfp4_skinny_workspace_bytes(4, 4096, 14336) == before
    assert lib.ac4k_set_linear_tuning(0, 0, 0, 0, 0) == 0
    assert lib.ac4k_debug_last_quantize_path() in (0, 1, 2, 3)
    # K <= 0 never selects a weight-streaming plan, and the workspace entry points say what is wrong
    assert lib.ac4k_linear_nvfp4_skinny_workspace_bytes(8, 1024, 0) == 0
    assert lib.ac4k_linear_nvfp4_skinny_workspace_bytes(8, 1024, -256) == 0
    rc = lib.ac4k_linear_nvfp4_skinny(one, 0, one, one, one, one, one, one, None, 0, 8, 1024, 0, one, 256, None)
    assert rc != 0 and b"positive" in lib.ac4k_last_error()
    rc = lib.ac4k_linear_nvfp4_skinny_static(one, 0, one, one, one, one, one, one, None, 0, 8, 1024, -256, None)
    assert rc != 0 and b"positive" in lib.ac4k_last_error()
    rc = lib.ac4k_linear_nvfp4_fused_bf16(one, 0, one, one, one, one, one, one, one, None, 0, 8, 1024, 0, one, 256, None)
    assert rc != 0 and b"positive" in lib.ac4k_last_error()
    rc = lib.ac4k_linear_nvfp4_fused_bf16(one, 0, one, one, one, one, one, one, one, None, 0, 64, 4, 64, one, 0, None)
    assert rc != 0 and b"1 <= M <= 32" in lib.ac4k_last_error()
    with pytest.raises(RuntimeError):
        _lib.check(rc)


def test_python_checks_without_gpu():
    import torch
    from ac4k_kernel_amd import ops
    x = torch.zeros((4, 64), dtype=torch.bfloat16)
    with pytest.raises(AssertionError):
        ops.quantize(x, 0, 0)
    with pytest.raises(AssertionError):
        ops.quantize(x, 0, 1, precision="fp4")
    with pytest.raises(AssertionError):
        ops.quantize(torch.zeros(8, dtype=torch.bfloat16), 0, 1)
    with pytest.raises(RuntimeError):  # CPU tensor: "must be a CUDA tensor"
        ops.quantize_fp8(torch.empty((4, 64), dtype=torch.float8_e4m3fn), torch.empty(16), x,
                         torch.tensor(448.0), 0, 1, False)


def test_reference_import_lines_resolve():
    """The import lines of the reference's callers (test/test_quantize_bench.py:7,
    test/test_linear_bench.py:4) resolve to this library through the `ac4k_kernel` alias package."""
    import ac4k_kernel
    import ac4k_kernel_amd
    from ac4k_kernel.ops import attention, linear, quantize
    from ac4k_kernel.ops.attention import mha_int8_x_fp8_fwd, mha_nvfp4_fwd
    from ac4k_kernel.ops.linear import Ac4kLinearOp
    from ac4k_kernel.ops.quant import Ac4kQuantizeOp
    import ac4k_kernel._rocm_ops as binding
    assert ac4k_kernel.get_backend() == "rocm" and ac4k_kernel.get_arch() == "gfx950"
    assert ac4k_kernel.get_info() == ac4k_kernel_amd.get_info()
    assert quantize is ac4k_kernel_amd.ops.quantize and linear is ac4k_kernel_amd.ops.linear
    assert attention is ac4k_kernel_amd.ops.attention and mha_nvfp4_fwd is binding.mha_nvfp4_fwd
    assert mha_int8_x_fp8_fwd is binding.mha_int8_x_fp8_fwd
    assert binding is ac4k_kernel_amd._rocm_ops and binding.__backend__ == "rocm"
    assert issubclass(Ac4kLinearOp, __import__("torch").nn.Module) and Ac4kQuantizeOp is not None
    for name in ("quantize_nvfp4", "quantize_fp8", "quantize_int8", "linear_nvfp4"):
        assert getattr(ac4k_kernel, name) is getattr(ac4k_kernel_amd, name)
        assert getattr(ac4k_kernel.ops, name) is getattr(ac4k_kernel_amd.ops, name)
    # the alias must not pull in the checker either
    for f in ("__init__.py", os.path.join("ops", "__init__.py")):
        assert "oracle" not in open(os.path.join(ROOT, "ac4k_kernel", f)).read()


@pytest.mark.parametrize("B,H,Nq,Nkv,D,Dv", [(4096, 12, 64, 64, 64, 64), (65535, 12, 49, 49, 32, 32), (1024, 3, 256, 256, 40, 128),
                                             (2, 12, 777, 257, 64, 64), (1, 1, 40, 9000, 8, 128), (1, 40, 16384, 16384, 128, 128)])
def test_attention_workspace_is_no_larger_than_the_separate_operators(B, H, Nq, Nkv, D, Dv):
    """The whole INT8 x FP8 call keeps the quantized operands and partial results; operator by operator the same operands lie
    beside a bf16 copy of K (less its mean), so whatever fits there fits here."""
    from ac4k_kernel_amd import _lib
    up = lambda a, b: -(-a // b) * b  # noqa: E731
    operands = Nq * up(D, 16) + Nkv * up(D, 16) + Dv * up(Nkv, 16) + 4 * (-(-Nq // 64) - (-Nkv // 128) + up(Dv, 16))
    k_copy = 2 * Nkv * D
    got = _lib.load().ac4k_attention_int8_x_fp8_workspace_bytes(B, H, Nq, Nkv, D, Dv)
    assert B * H * operands <= got <= B * H * (operands + k_copy) + 8 * 256  # eight buffers, 256-byte aligned


def test_whole_attention_leaves_head_counts_beyond_a_launch_to_the_separate_operators():
    """2^24 workgroups of 256 threads are 2^32 threads: a launch does not carry them, so the whole calls do not take the sizes."""
    from ac4k_kernel_amd import _lib
    lib = _lib.load()
    for f in (lib.ac4k_attention_int8_x_fp8_workspace_bytes, lib.ac4k_attention_nvfp4_workspace_bytes):
        assert f(1024, 5461, 1, 1, 16, 16) > 0   # three workgroups a head: 2^24 - 1024
        assert f(4096, 2049, 1, 1, 16, 16) == -1


@pytest.mark.parametrize("m,n,k", [(16, 4096, 14336), (16, 4096, 14400), (100, 5003, 2816), (100, 5003, 2880), (300, 256, 4160)])
def test_linear_workspace_is_checked(m, n, k):
    from ac4k_kernel_amd import _lib
    lib, p = _lib.load(), ctypes.c_void_p(256)  # never dereferenced
    need = lib.ac4k_linear_nvfp4_workspace_bytes(m, n, k)
    assert need > 0
    call = lambda ws, size: lib.ac4k_linear_nvfp4_workspace(p, 0, p, p, p, p, p, p, None, 0, m, n, k, ws, size, None)  # noqa: E731
    for ws, size, text in ((p, need - 1, b"too small"), (None, need, b"256-byte aligned"), (ctypes.c_void_p(272), need, b"256-byte aligned")):
        assert call(ws, size) != 0 and text in lib.ac4k_last_error()


def test_attention_operands_and_workspace_are_checked():
    """Dense [1, 2, 64, 64] operands, in either layout, and what the whole calls refuse about them."""
    from ac4k_kernel_amd import _lib
    lib, p = _lib.load(), ctypes.c_void_p(256)  # never dereferenced
    size = (1, 2, 64, 64, 64, 64)
    for entry, bytes_, scale in ((lib.ac4k_attention_int8_x_fp8_bf16, lib.ac4k_attention_int8_x_fp8_workspace_bytes, 2.25),
                                 (lib.ac4k_attention_nvfp4_bf16, lib.ac4k_attention_nvfp4_workspace_bytes, 2688.0)):
        need, dense = bytes_(*size), (8192, 4096, 64)

        def call(q=dense, k=dense, v=dense, ptr=p, size=size, ws=p, ws_bytes=need):
            return entry(p, 8192, 4096, 64, 1, ptr, *q, p, *k, p, *v, *size, scale, 0.125, ws, ws_bytes, None)

        for kw, text in (({"ws_bytes": need - 1}, b"too small"), ({"ws": ctypes.c_void_p(264)}, b"16-byte aligned"), ({"ptr": None}, b"null"),
                         ({"ptr": ctypes.c_void_p(257)}, b"2-byte aligned"), ({"k": (8192, -64, 64)}, b"negative"),
                         ({"size": (1, 2, 64, 64, 64, 136)}, b"8 to 128"), ({"size": (1, 2, 0, 64, 64, 64)}, b"positive")):
            assert call(**kw) != 0 and text in lib.ac4k_last_error(), (kw, lib.ac4k_last_error())
        assert bytes_(1, 2, 64, 64, 7, 64) == -1 and bytes_(1, 2, 64, 64, 64, 129) == -1 and bytes_(0, 2, 64, 64, 64, 64) == -1
    for gap in ((8192, 4096, 65), (8192, 4097, 64)):  # the NVFP4 maxima are taken over whole tensors
        assert call(k=gap) != 0 and b"dense" in lib.ac4k_last_error()


def test_scratch_sizes_of_every_plan_without_gpu():
    """The sizes are pure functions of the shape: decode-sized, K-split and tile plans answer without a GPU, and what a linear
    allocates is nothing or all of what the workspace entry point insists on.  Sizes that callers may have kept, and which of
    them are not allocated: a plan of one K range, a 16-row kernel, and (all of it) a plan that writes half of what it asks for."""
    from ac4k_kernel_amd import _lib
    lib = _lib.load()
    for m in (1, 2, 8, 16, 17, 32, 33, 64, 100, 128, 129, 200, 300, 1001, 4096):
        for n in (1, 128, 1000, 4096, 14336, 28672, 65536):
            for k in (64, 256, 320, 1024, 2880, 4096, 14336):
                asked = lib.ac4k_linear_nvfp4_workspace_bytes(m, n, k)
                assert lib.ac4k_linear_nvfp4_scratch_bytes(m, n, k) in (0, asked)
                assert lib.ac4k_linear_nvfp4_prepacked_workspace_bytes(m, n, k) >= 0
    sizes = [lib.ac4k_linear_nvfp4_workspace_bytes(*s) for s in ((512, 4096, 14336), (150, 4096, 4096), (16, 4096, 14336))]
    assert sizes == [33554432, 9830400, 1048576]
    for shape, asked, taken in (((512, 4096, 14336), 33554432, 33554432), ((200, 4096, 4096), 13107200, 13107200), ((300, 4096, 4096), 9830400, 0),
                                ((16, 4096, 14336), 1048576, 0), ((3, 337, 14336), 226464, 226464), ((64, 1024, 4096), 2097152, 2097152),
                                ((2048, 14336, 4096), 0, 0), ((300, 4096, 4112), 0, 0)):
        assert (lib.ac4k_linear_nvfp4_workspace_bytes(*shape), lib.ac4k_linear_nvfp4_scratch_bytes(*shape)) == (asked, taken), shape


def test_a_linear_asks_for_its_scratch_once(monkeypatch):
    """One size query per linear, whose answer is the size of the scratch."""
    import torch
    from ac4k_kernel_amd import _lib, _rocm_ops
    lib, asked, launched = _lib.load(), [], []

    class Counting:
        def __getattr__(self, name):
            f = getattr(lib, name)
            if name.endswith("_bytes"):
                return lambda *a: asked.append((name, f(*a))) or asked[-1][1]
            return lambda *a: launched.append((name, a)) or 0

    class OnGpu(torch.Tensor):  # passes the device checks; nothing is launched on it
        is_cuda = True

    monkeypatch.setattr(_rocm_ops, "_L", Counting())
    monkeypatch.setattr(_rocm_ops, "_stream", lambda: 0)
    t = lambda shape, dtype: torch.zeros(shape, dtype=dtype).as_subclass(OnGpu)  # noqa: E731
    for m, n, k, size in ((64, 1024, 4096, 2097152), (200, 4096, 4096, 13107200), (16, 1024, 2048, 0)):
        asked.clear(), launched.clear()
        gs = t((), torch.float32)
        operand = lambda rows: (t((rows, k // 2), torch.uint8), t((k // 64, -(-rows // 16) * 16, 4), torch.float8_e4m3fn), gs)  # noqa: E731
        _rocm_ops.linear_nvfp4(t((m, n), torch.bfloat16), *operand(m), *operand(n))
        assert [size] == [b for _, b in asked] and len(launched) == 1
        name, args = launched[0]
        assert (name, args[-2]) == (("ac4k_linear_nvfp4_workspace", size) if size else ("ac4k_linear_nvfp4", k))


@pytest.mark.parametrize("precision", ["int8+fp8e4m3", "nvfp4"])
@pytest.mark.parametrize("which", ["q", "k", "v", "out"])
def test_attention_refuses_operands_that_are_not_4d(precision, which):
    import torch
    from ac4k_kernel_amd import ops
    t = {name: torch.zeros((2, 64, 4, 64), dtype=torch.bfloat16) for name in ("q", "k", "v", "out")}
    t[which] = t[which][0]
    with pytest.raises(RuntimeError):
        ops.attention(t["q"], t["k"], t["v"], out=t["out"], layout="BNHD", precision=precision)


def decode_kernel(m, n, k):
    from ac4k_kernel_amd import _lib
    launches = ctypes.c_int(-1)
    return _lib.load().ac4k_debug_linear_decode_kernel(m, n, k, ctypes.byref(launches)), launches.value


@pytest.mark.parametrize("m,k", [(1, 256), (1, 512), (1, 2048), (4, 256), (16, 256), (16, 320), (32, 256), (16, 2880)])
def test_sixteen_row_workgroups_stay_within_a_launch(m, k):
    """512 threads for 16 weight rows: 2^23 workgroups are 2^32 threads, more than a launch carries, and no error when it drops them."""
    assert decode_kernel(16, 4096, 256) == (4, 1) and decode_kernel(16, 4096, 14336) == (4, 2) and decode_kernel(64, 4096, 4096) == (0, 0)
    for n in (2 ** 27 - 15, 2 ** 27 - 8, 2 ** 27 - 1, 2 ** 27):
        kernel, launches = decode_kernel(m, n, k)
        assert kernel not in (4, 5) and launches != 1, n
    assert decode_kernel(16, 2 ** 27 - 16, 256)[0] == 4  # the last that a launch carries


def test_sixteen_row_workgroups_on_an_image_where_they_are_faster():
    """M above 16, where the ring (2) was taken from shapes on which 16-row workgroups (4) are 4 to 18 % slower, and others that they are faster on."""
    from ac4k_kernel_amd import _lib
    f = _lib.load().ac4k_debug_linear_prepacked_decode_kernel
    for shape in ((31, 320, 14080), (29, 22656, 512), (22, 384, 13568), (28, 384, 12672), (26, 888, 13312), (31, 19840, 512)):
        assert f(*shape) == 2, shape
    for shape in ((24, 4096, 8192), (24, 4112, 2048), (32, 4096, 14336), (20, 12288, 12288), (32, 128, 2048), (16, 4096, 14336), (1, 28672, 8192)):
        assert f(*shape) == 4, shape
    assert f(33, 4096, 4096) == 0 and f(16, 4096, 128) == 0


def test_fused_calls_and_linears_sum_alike():
    """A fused call in one launch sums as the 16-row kernels do, so a linear of the same shape runs one of them: the two are equal bit
    for bit.  Shapes of one launch are among all of these sizes."""
    one = 0
    for m in (1, 2, 3, 4, 5, 8, 16, 17, 32):
        for n in (1, 16, 130, 384, 512, 1024, 1536, 4096, 8192, 14336, 24576, 28672, 65536):
            for k in (256, 512, 768, 1024, 2048, 4096, 5376, 8192, 10240, 12288, 14336, 16384):
                kernel, launches = decode_kernel(m, n, k)
                one += launches == 1
                assert launches in (1, 2, 3) and (launches != 1 or kernel in (4, 5)) and (kernel != 5 or m <= 16), (m, n, k)
    assert one > 300
    for shape in ((1, 28672, 8192), (2, 28672, 8192), (1, 24576, 10240), (1, 512, 8192), (1, 1024, 16384)):
        assert decode_kernel(*shape) == (5, 1)
    assert decode_kernel(1, 4096, 4096) == (4, 1)
