"""CPU-side checks: the C-ABI library loads and exports every declared symbol,
argument validation raises the reference's exception types before any GPU work,
and the torch-level entry points agree with the oracle."""
import ctypes
import os
import re

import pytest
import torch

import oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    from approx_topk import _native
    header = open(os.path.join(ROOT, "include", "approx_topk_hip.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(atk_[a-z0-9_]+)\s*\(", header))
    assert {"atk_version", "atk_strerror", "atk_stage1", "atk_select", "atk_topk"} <= declared
    handle = ctypes.CDLL(_native.library_path())
    for name in declared:
        assert hasattr(handle, name), name
    assert set(_native._SIGNATURES) == declared
    # the clock stamps of the phase timelines (csrc/atk_trace.h) exist only in a library built for them
    assert not hasattr(handle, "atk_trace_fused_row_f16") and not hasattr(handle, "atk_trace_stage1_stream_f32")
    assert _native.lib().atk_version() == _native.ABI_VERSION
    assert _native.lib().atk_strerror(0) == b"ok"
    assert b"j must" in _native.lib().atk_strerror(-2)


def test_workspace_of_one_call_depends_on_the_address():
    from approx_topk import _native
    L = _native.lib()
    # 512 fp16 rows of 32768, 1024 candidates: one kernel, nothing parked
    general = L.atk_topk_workspace_bytes(512, 32768, 1024, 1, 256, 0, 1)
    assert general >= 512 * 1024 * (2 + 8)
    assert L.atk_topk_workspace_bytes_at(4096, 512, 32768, 32768, 1024, 1, 256, 0, 1) == 0
    # rows off 16 bytes keep the bound of two kernels, whatever takes them
    assert L.atk_topk_workspace_bytes_at(4098, 512, 32768, 32768, 1024, 1, 256, 0, 1) == general
    assert L.atk_topk_workspace_bytes_at(4096, 512, 32768, 32769, 1024, 1, 256, 0, 1) == general
    # k == k0: stage 1 alone
    assert L.atk_topk_workspace_bytes_at(4096, 512, 32768, 32768, 1024, 1, 1024, 0, 1) == \
        L.atk_topk_workspace_bytes(512, 32768, 1024, 1, 1024, 0, 1)
    # contiguous buckets: one kernel for buckets of up to 256 bytes (here 32 elements), else two
    assert L.atk_topk_workspace_bytes_at(4096, 512, 32768, 32768, 1024, 1, 256, 1, 1) == 0
    assert L.atk_topk_workspace_bytes_at(4096, 512, 1 << 18, 1 << 18, 1024, 1, 256, 1, 1) == \
        L.atk_topk_workspace_bytes(512, 1 << 18, 1024, 1, 256, 1, 1) > 0


def test_workspace_a_call_uses_follows_the_kernels_it_takes():
    from approx_topk import _native
    L = _native.lib()

    def used(x, n, stride, k0, j, k, layout=0, code=1):
        args = (512, n, stride, k0, j, k, layout, code)
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(x, *args, 4096, 4096, buf, 1024) == 0
        need = L.atk_topk_workspace_bytes_used(x, *args)
        assert need <= L.atk_topk_workspace_bytes_at(x, *args) <= L.atk_topk_workspace_bytes(512, n, *args[3:])
        one_kernel = buf.value.startswith(b"fused_")
        assert (need == 0) == one_kernel and need in (0, L.atk_topk_workspace_bytes(512, n, *args[3:]))
        return one_kernel

    assert used(4096, 32768, 32768, 1024, 1, 256)
    for n, stride in ((32768, 32769), (32768, 32775), (32767, 32767), (32761, 32768)):   # rows that start anywhere
        assert used(4096, n, stride, 1024, 1, 256) and used(4100, n, stride, 1024, 1, 256)
        assert used(4098, n, stride, 1024, 1, 256)            # ... on an odd half-word as well
    assert used(4098, 32768, 32768, 1024, 1, 256)
    assert not used(4096, 32768, 32768, 1022, 2, 511)         # a number of buckets off the load width
    assert used(4096, 32768, 32768, 1024, 1, 256, layout=1) and not used(4096, 1 << 18, 1 << 18, 1024, 1, 256, layout=1)
    # what no kernel takes needs none of its own: the bound, as for every invalid call
    assert L.atk_topk_workspace_bytes_used(4096, 0, 32768, 32768, 1024, 1, 256, 0, 1) == 0
    # the operator's wrapper allocates by it
    assert _native._topk_workspace(0, 512, 32768, 32769, 1024, 1, 256, 0, 1) == 0
    assert _native._topk_workspace(2, 512, 32768, 32768, 1024, 1, 256, 0, 1) == 0
    assert _native._topk_workspace(0, 512, 32768, 32768, 1022, 2, 511, 0, 1) > 0


def test_native_argument_checks_need_no_gpu():
    # rejected before any launch, so callable here
    from approx_topk import _native
    L = _native.lib()
    buf = ctypes.create_string_buffer(64)
    p = ctypes.addressof(buf)
    assert L.atk_stage1(p, 1, 8, 8, 6, 4, 0, 0, p, p, None, 0, None) == -2     # j does not divide k0
    assert L.atk_stage1(p, 1, 8, 8, 5, 5, 0, 0, p, p, None, 0, None) == -2     # j out of range
    assert L.atk_stage1(p, 1, 8, 8, 16, 1, 0, 0, p, p, None, 0, None) == -3    # k0 > n
    assert L.atk_stage1(p, 1, 8, 8, 4, 1, 9, 0, p, p, None, 0, None) == -4     # layout
    assert L.atk_stage1(p, 1, 8, 8, 4, 2, 2, 0, p, p, None, 0, None) == -4     # padded layout, j != 1
    assert L.atk_stage1(p, 1, 8, 8, 4, 1, 0, 99, p, p, None, 0, None) == -1    # dtype
    assert L.atk_stage1(None, 1, 8, 8, 4, 1, 0, 0, p, p, None, 0, None) == -7  # null input
    assert L.atk_stage1(p, 1, 8, 4, 4, 1, 0, 0, p, p, None, 0, None) == -7     # row_stride < n
    assert L.atk_stage1(p, 1, 8, 8, 0, 1, 0, 0, p, p, None, 0, None) == 0      # k0 == 0: no-op
    assert L.atk_topk(p, 1, 1 << 20, 1 << 20, 4, 1, 2, 0, 0, p, p, None, 0, None) == -5    # workspace missing (two kernels)
    assert L.atk_topk(p, 1, 8, 8, 4, 1, 5, 0, 0, p, p, None, 0, None) == -3    # k > k0
    assert L.atk_select(p, p, 1, 4, 5, 8, 0, p, p, None, 0, None) == -3
    # misaligned pointers: data to the element size, indices to their width, workspace to 16 bytes
    assert p % 16 == 0
    assert L.atk_stage1(p + 2, 1, 8, 8, 4, 1, 0, 0, p, p, None, 0, None) == -9      # fp32 input at +2
    assert L.atk_stage1(p, 1, 8, 8, 4, 1, 0, 0, p + 1, p, None, 0, None) == -9      # values
    assert L.atk_stage1(p, 1, 8, 8, 4, 1, 0, 0, p, p + 4, None, 0, None) == -9      # int64 indices at +4
    assert L.atk_stage1_i32(p, 1, 8, 8, 4, 1, 0, 0, p, p + 2, None, 0, None) == -9  # int32 indices at +2
    assert L.atk_stage1(p, 1, 8, 8, 4, 1, 0, 0, p, p, p + 8, 64, None) == -9        # workspace at +8
    assert L.atk_topk(p, 1, 1 << 20, 1 << 20, 4, 1, 2, 0, 0, p, p, p + 8, 1 << 30, None) == -9
    assert L.atk_select(p, p + 4, 1, 4, 2, 8, 0, p, p, None, 0, None) == -9         # candidate indices
    assert L.atk_select(p, p, 1, 4, 2, 8, 0, p, p, p + 4, 1 << 20, None) == -9
    assert b"misaligned" in L.atk_strerror(-9)
    assert L.atk_topk_workspace_bytes(3, 100, 8, 1, 8, 0, 0) == 0
    assert L.atk_topk_workspace_bytes(3, 100, 16, 1, 8, 0, 0) >= 3 * 16 * 12


def test_describe_names_the_planned_kernels():
    # the planner's choice for a call, as text (no GPU needed: nothing is enqueued)
    from approx_topk import _native
    L = _native.lib()

    def describe(rows, n, code, k, j, k_mult, x=4096):
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(x, rows, n, n, k * k_mult, j, k, 0, code, 4096, 4096, buf, 1024) == 0
        return buf.value.decode()
    c2 = describe(128, 1 << 20, 0, 65536, 2, 1)
    assert c2.startswith("stream_kernel<f32, J=2, V=4, W=8, U=8, RUN=4, PACKED=0> grid=16384 block=512")
    c3 = describe(1024, 32768, 1, 2048, 4, 4)
    assert c3.startswith("fused_regs_kernel<f16, J=4, V=4, pos16, PACKED=1> grid=1024 block=512")
    c5 = describe(1, 1 << 26, 0, 16384, 4, 2)
    assert c5.startswith("stream_kernel<f32, J=4") and "stream_merge_kernel" in c5 and "chain_solo_kernel" in c5
    # few buckets (narrow sub-rows): the streaming kernel, which folds sub-rows side by side,
    # not the one-kernel path, whose lanes would idle; short rows of few sub-rows stay with it
    assert describe(256, 1 << 22, 1, 4, 1, 2).startswith("stream_kernel<f16, J=1")
    assert describe(4, 32768, 1, 4, 2, 2).startswith("stream_kernel<f16, J=2")
    assert describe(4, 32768, 0, 4, 4, 8).startswith("stream_kernel<f32, J=4")
    assert describe(64, 1024, 1, 8, 1, 2).startswith("fused_regs_kernel<f16, J=1")
    # the select over several workgroups per row: few rows only, one launch up to 32768 candidates
    assert "chain_solo_kernel<f32> grid=16 " in describe(1, 1 << 24, 0, 8192, 2, 2)
    assert "chain_emit_kernel<f32> grid=512 block=256 per_thread=4" in describe(8, 1 << 22, 0, 32768, 2, 2)
    # more rows of more than 32768 candidates: segments of 4096 candidates; beyond 64 rows other selects
    assert "chain_emit_kernel<f32> grid=2048 block=256 per_thread=16" in describe(64, 1 << 18, 0, 16384, 2, 8)
    assert "chain_" not in describe(65, 1 << 18, 0, 16384, 2, 8)
    assert "chain_" not in describe(17, 1 << 20, 0, 16384, 1, 2)
    # an input that starts on an odd half-word is loaded like rows that do
    assert describe(1024, 32768, 1, 2048, 4, 4, x=4098) == c3
    # contiguous buckets of 16-256 bytes with a second stage: one kernel too; longer buckets, a bucket
    # count that does not fill whole column tiles, or a row with a remainder: two kernels
    def contiguous(rows, n, code, k, j, k_mult):
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, rows, n, n, k * k_mult, j, k, 1, code, 4096, 4096, buf, 1024) == 0
        return buf.value.decode()
    short = contiguous(1024, 32768, 1, 2048, 4, 4)
    assert short.startswith("fused_regs_kernel<f16, J=4, V=4, pos16, PACKED=1> grid=1024 block=512")
    assert short.endswith("short contiguous buckets") and "select" not in short
    assert contiguous(1024, 32768, 0, 2048, 4, 4).endswith("short contiguous buckets")   # fp32: 64 bytes
    assert contiguous(1024, 65536, 0, 2048, 4, 4).endswith("short contiguous buckets")   # 128 bytes
    assert contiguous(256, 1 << 18, 0, 2048, 4, 4).startswith("contig_kernel<f32")        # 512 bytes
    # no second stage: a lane per bucket up to 64 bytes, spans of buckets through LDS beyond
    assert contiguous(1024, 32768, 1, 2048, 4, 1).startswith("contig_kernel<f16")         # 128 bytes
    assert contiguous(1024, 32768, 1, 4096, 4, 1).startswith("whole_bucket_kernel<f16, J=4> grid=4096 block=256")
    assert contiguous(16384, 1024, 1, 64, 2, 1).startswith("whole_bucket_kernel<f16, J=2> grid=2048 ")
    assert contiguous(16, 1028, 0, 256, 1, 1).startswith("contig_kernel<f32")             # 1028 = 4 * 256 + 4
    two = contiguous(16, 3072, 1, 64, 2, 4)                                               # 128 buckets: two kernels
    assert two.startswith("whole_bucket_kernel<f16, J=2> grid=8 ") and "select_kernel<f16" in two
    assert contiguous(16, 8200, 1, 512, 2, 2).startswith("contig_kernel<f16")             # 8200 = 16 * 512 + 8
    assert contiguous(1024, 32768, 4, 2048, 4, 4).startswith("contig_kernel<u8")          # 1-byte elements
    # truncation and argument checks
    buf = ctypes.create_string_buffer(8)
    assert L.atk_describe(4096, 128, 1 << 20, 1 << 20, 65536, 2, 65536, 0, 0, 4096, 4096, buf, 8) == 0
    assert buf.value == b"stream_"
    assert L.atk_describe(4096, 1, 8, 8, 6, 4, 6, 0, 0, 4096, 4096, buf, 8) == -2


def test_validation_errors_before_device_check():
    from approx_topk import topk
    x = torch.randn(8, 64)
    with pytest.raises(NotImplementedError):
        topk(x, 4, 0, j=2)
    with pytest.raises(ValueError):
        topk(x, 4, -1, k_mult=0)
    with pytest.raises(RuntimeError, match="j must divide k"):
        topk(x, 6, -1, j=4)
    with pytest.raises(RuntimeError, match="0 < j < 5"):
        topk(x, 5, -1, j=5)
    with pytest.raises(RuntimeError, match="k must not be larger"):
        topk(x, 128, -1)
    with pytest.raises(RuntimeError, match="GPU"):
        topk(x, 4, -1)          # valid arguments, but no CPU path exists
    v, i = topk(x, 0, -1, j=0)  # k == 0 is valid and does no work
    assert v.shape == (8, 0) and i.dtype == torch.int64


def test_fake_impl_shapes():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from approx_topk import topk
    with FakeTensorMode():
        x = torch.empty(5, 32, 512)
        v, i = topk(x, 64, -1, j=2, k_mult=2)
        assert v.shape == (5, 32, 64) and i.shape == (5, 32, 64)
        assert v.dtype == torch.float32 and i.dtype == torch.int64


def test_topk_torch_known_answers_and_oracle():
    from approx_topk.experimental.bucketed_argmax import topk_torch
    x = torch.stack([100 * torch.arange(0, 20), -100 * torch.arange(0, 20)]).float()
    v, i = topk_torch(x, k=3, dim=1, interleaved=False)
    assert v.tolist() == [[600.0, 1300, 1900], [0, -700, -1400]] and i.tolist() == [[6, 13, 19], [0, 7, 14]]
    vt, it = topk_torch(x.T, k=3, dim=0, interleaved=False)
    assert torch.equal(vt.T, v) and torch.equal(it.T, i)
    v, i = topk_torch(x, k=3, dim=1, interleaved=True)
    assert v.tolist() == [[1800.0, 1900, 1700], [0, -100, -200]] and i.tolist() == [[18, 19, 17], [0, 1, 2]]
    g = torch.Generator().manual_seed(1001)
    c1 = torch.randn(4, 65536, generator=g)
    for interleaved in (True, False):
        v, i = topk_torch(c1, 1024, -1, interleaved)
        ev, ei = oracle.bucketed_argmax(c1, 1024, -1, interleaved)
        assert torch.equal(v, ev) and torch.equal(i, ei)


def test_batch_contiguous():
    from approx_topk.experimental.bucketed_argmax import _batch_contiguous
    x = torch.arange(3 * 4 * 5).view(3, 4, 5)
    for t, same in [(x, True), (x[:, :, :-1], True), (x[:, :, ::2], False), (x[:, :-1, :], False),
                    (x.swapdims(0, 1), False)]:
        t2 = _batch_contiguous(t)
        assert (t2 is t) == same
        assert torch.equal(t, t2)
        if not same:
            assert t2.is_contiguous()


def test_rows_view():
    from approx_topk import _native
    x = torch.arange(3 * 4 * 10.0).view(3, 4, 10)
    t, rows, n, step = _native.rows_view(x)
    assert t is x and (rows, n, step) == (12, 10, 10)
    t, rows, n, step = _native.rows_view(x[:, :, :7])
    assert t.data_ptr() == x.data_ptr() and (rows, n, step) == (12, 7, 10)
    t, rows, n, step = _native.rows_view(x[:, :3, :])
    assert t.is_contiguous() and (rows, n, step) == (9, 10, 10)
    t, rows, n, step = _native.rows_view(x.movedim(1, -1))
    assert t.is_contiguous() and (rows, n, step) == (30, 4, 4)



def test_operator_object_offers_register_fake_and_register_autograd():
    # the reference's `topk` is a CustomOpDef with these two methods (priority_queue.py:14,91); in a child
    # process, because both registrations change the operator for everything that runs after them
    import subprocess
    import sys
    import textwrap

    code = textwrap.dedent("""
        import sys
        sys.path.insert(0, %r)
        import torch
        from torch._subclasses.fake_tensor import FakeTensorMode
        from approx_topk import topk

        @topk.register_fake
        def _(xs, k, dim, j=None, k_mult=1, interleaved=True, multithread_buckets=False):
            shape = list(xs.shape)
            shape[dim] = k
            return xs.new_empty(shape), xs.new_empty(shape, dtype=torch.int64)

        with FakeTensorMode():
            v, i = topk(torch.empty(3, 64), 8, -1, 2, 1)
        assert tuple(v.shape) == (3, 8) and i.dtype == torch.int64

        def setup(ctx, inputs, output):
            ctx.save_for_backward(output[1])
            ctx.shape = inputs[0].shape

        def backward(ctx, grad_values, grad_indices):
            (indices,) = ctx.saved_tensors
            return torch.zeros(ctx.shape).scatter(-1, indices, grad_values), None, None, None, None, None, None

        topk.register_autograd(backward, setup_context=setup)
        print("registered")
    """) % os.path.join(ROOT, "pytorch-approx-topk_amd")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "registered" in out.stdout, out.stderr[-2000:]


def test_gradient_operator_checks_its_tensors_before_any_native_call():
    # the kernel reads rows * k entries of both tensors, the indices eight bytes each: what does not
    # match must not reach it
    op = torch.ops.approx_topk.topk_grad.default
    w, i = torch.randn(3, 8), torch.zeros(3, 8, dtype=torch.int64)
    with pytest.raises(RuntimeError, match="GPU"):
        op(w, i, 64, 8, 1, True)                       # valid arguments, but no CPU path exists
    for grad_values, indices in ((w, i.int()), (w, i.double()), (w[:2], i), (w[:, :4], i), (w[0], i), (w, i[0]),
                                 (w.reshape(8, 3), i), (w, i.to("meta")), (w[0, 0], i[0, 0])):
        with pytest.raises(RuntimeError, match="topk_grad"):
            op(grad_values, indices, 64, 8, 1, True)


def test_no_kernel_of_a_contiguous_call_has_more_threads_than_a_launch_takes():
    # 32 bits count them; batches beyond that many lanes keep the kernel that needs fewer
    from approx_topk import _native
    L = _native.lib()

    def describe(rows, n, code, k, j):
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, rows, n, n, k, j, k, 1, code, 4096, 4096, buf, 1024) == 0
        return buf.value.decode()

    for rows, n, code, k, j in ((16260510, 2803, 0, 292, 2), (12075969, 3677, 0, 106, 1), (16275156, 2318, 7, 54, 3)):
        text = describe(rows, n, code, k, j)
        grid, block = (int(re.search(f"{key}=(\\d+)", text).group(1)) for key in ("grid", "block"))
        assert grid * block < 1 << 32, text
    # two lanes to each of 146 buckets: 2^24 - 1 workgroups of 256 are the most
    assert describe(14708791, 2803, 0, 292, 2).startswith("split_bucket_kernel<f32")
    assert describe(14708792, 2803, 0, 292, 2).startswith("contig_kernel<f32")


# (type code, rows, n, k, j, k_mult): calls timed with 16-byte and with one-element loads in one-stage and two-stage
# kernels, at least 15 % apart: the planner takes the faster one
NARROW = [
    (0, 39, 761703, 40, 2, 1), (0, 16, 110067, 112, 2, 1), (0, 5, 119152, 572, 2, 1), (0, 5, 432090, 108, 3, 2),
    (7, 17, 56249, 388, 4, 1), (7, 2, 1096704, 1764, 2, 1), (7, 1, 1896432, 64458, 2, 1),
    (1, 5, 41786, 592, 4, 1), (2, 14, 75102, 424, 4, 1), (1, 10, 98448, 154, 2, 2), (2, 11, 3395763, 1088, 2, 1),
    (1, 3, 15355401, 572, 4, 2),
    (5, 1, 172601, 5240, 4, 1), (5, 1, 2514382, 20604, 4, 1), (5, 33, 511713, 1845, 3, 1), (5, 85, 84195, 520, 2, 1),
    (4, 39, 152696, 804, 4, 1), (4, 26, 379453, 2120, 2, 1), (4, 5, 1954268, 525, 3, 1),
    (3, 6, 108793, 1833, 3, 1), (3, 2, 310384, 3196, 4, 1), (8, 1, 112815, 1752, 4, 1), (8, 14, 71905, 112, 2, 1),
]
WIDE = [
    (0, 71, 276112, 4172, 2, 1), (0, 128, 1 << 20, 65536, 2, 1),
    (2, 3011, 15788, 1500, 3, 1), (1, 21, 1426304, 16676, 2, 1), (1, 65, 303684, 2924, 2, 1), (2, 17, 847929, 82694, 1, 1),
    (6, 4, 12701536, 102288, 4, 1), (6, 26, 602919, 495, 1, 1), (2, 98, 1 << 19, 1024, 2, 2),
    (5, 51, 507136, 7173, 3, 1), (4, 236, 122243, 220, 2, 4), (4, 51, 2066190, 7404, 3, 2),
]


@pytest.mark.parametrize("vec,calls", [("V=1,", NARROW), ("wide", WIDE)], ids=["narrow", "wide"])
def test_the_width_of_loads_follows_the_faster_plan(vec, calls):
    from approx_topk import _native
    L = _native.lib()
    for code, rows, n, k, j, k_mult in calls:
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, rows, n, n, k * k_mult, j, k, 0, code, 4096, 4096, buf, 1024) == 0
        text = buf.value.decode()
        want = vec if vec != "wide" else f"V={min(8, 16 // [4, 2, 2, 8, 1, 1, 2, 4, 8][code])},"
        assert text.startswith("stream_kernel<") and want in text, (rows, n, k, j, k_mult, text)


def test_rows_of_one_byte_elements_on_8_bytes_are_rows_on_their_load_width():
    # (a load of theirs is 8 bytes: they were accepted by the one-kernel path, and by the call that cannot
    # allocate, before rows of any start were)
    from approx_topk import _native
    L = _native.lib()
    limit = 8 << 20
    for args in ((362, 18608, 18616, 4416, 3, 1104, 0, 5), (960, 16248, 16248, 3144, 3, 1572, 0, 5),
                 (154, 239560, 239576, 22304, 4, 11152, 0, 4), (4096, 8200, 8200, 1024, 1, 256, 0, 4)):
        rows, n, _, k0, j, k, layout, code = args
        assert L.atk_topk_workspace_bytes(rows, n, k0, j, k, layout, code) > limit
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, *args, 4096, 4096, buf, 1024) == 0 and buf.value.startswith(b"fused_"), buf.value
        assert L.atk_topk_workspace_bytes_at(4096, *args) == 0 == L.atk_topk_workspace_bytes_used(4096, *args)
        # rows on 4 bytes, and an input off 16, keep the bound of two kernels
        off = (rows, n, n + 12, *args[3:])
        assert L.atk_topk_workspace_bytes_at(4096, *off) > limit and L.atk_topk_workspace_bytes_at(4104, *args) > limit


# the same for rows off 16 bytes with a second stage, timed in one kernel and in two
ONE_KERNEL = [
    (8, 254, 2501, 36, 2, 8), (8, 3, 24169, 358, 1, 2), (3, 206, 5521, 116, 1, 2), (6, 760, 2813, 41, 1, 4),
    (6, 100, 7861, 184, 4, 4), (8, 137, 10039, 452, 4, 2), (1, 288, 15375, 60, 2, 8), (1, 75, 42783, 476, 2, 4),
    (1, 742, 9559, 33, 1, 8), (7, 3312, 2349, 126, 1, 2), (0, 307, 18439, 304, 2, 2), (4, 1354, 66483, 286, 1, 8),
    (7, 171, 121527, 3366, 3, 4), (3, 170, 93177, 560, 2, 8), (2, 256, 100003, 64, 1, 8), (6, 46, 72589, 714, 4, 8),
]
TWO_KERNELS = [
    (4, 11, 10433, 128, 4, 4), (4, 1538, 37707, 400, 4, 8), (7, 33, 2131, 56, 4, 2), (3, 14, 3303, 16, 4, 8),
    (5, 2, 92341, 784, 4, 8), (1, 5, 104575, 196, 2, 4), (7, 3, 35717, 196, 4, 8), (2, 4, 118981, 402, 3, 8),
    (1, 2, 122721, 2580, 1, 2), (2, 7, 2193, 16, 4, 4), (1, 168, 298475, 544, 4, 4), (1, 9, 6995, 32, 2, 2),
    (0, 37, 2557, 24, 3, 2), (6, 152, 394615, 2280, 4, 2), (1, 183, 340470, 152, 4, 8),
]


@pytest.mark.parametrize("kernel,calls", [("fused_", ONE_KERNEL), ("stream_kernel<", TWO_KERNELS)], ids=["one", "two"])
def test_rows_off_16_bytes_take_one_kernel_where_that_is_faster(kernel, calls):
    from approx_topk import _native
    L = _native.lib()
    for code, rows, n, k, j, k_mult in calls:
        buf = ctypes.create_string_buffer(1024)
        args = (rows, n, n, k * k_mult, j, k, 0, code)
        assert L.atk_describe(4096, *args, 4096, 4096, buf, 1024) == 0
        assert buf.value.decode().startswith(kernel), (args, buf.value)
        # the workspace follows, also where the rows are those of a wider matrix
        assert (L.atk_topk_workspace_bytes_used(4096, *args) == 0) == (kernel == "fused_")


def test_few_long_contiguous_buckets_with_long_queues_keep_workgroups_of_their_own():
    # (a lane of split_bucket_kernel goes through eight pieces and more of such a bucket, queue and all)
    from approx_topk import _native
    L = _native.lib()

    def kernel(rows, m, b, j, code):
        n = b * m + b // 2
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, rows, n, n, b * j, j, b * j, 1, code, 4096, 4096, buf, 1024) == 0
        return buf.value.decode().split("_kernel")[0]

    for code in (0, 7):
        assert kernel(4, 7169, 32, 4, code) == kernel(1, 4353, 32, 3, code) == kernel(512, 16129, 1, 4, code) == "contig"
        assert kernel(32, 7169, 32, 4, code) == kernel(4, 4001, 32, 4, code) == "split_bucket"     # many; fewer pieces
        assert kernel(4, 7169, 32, 2, code) == "split_bucket"                                       # short queues
    for code in (1, 2, 6):
        assert kernel(4, 14337, 32, 4, code) == kernel(1, 8705, 32, 3, code) == "split_bucket"      # 16-bit elements


def test_no_plan_has_more_threads_than_a_launch_takes():
    # batches of very many short rows: one-element loads would take several times the workgroups, and the
    # second stage's of their own several times the threads of one kernel for both
    from approx_topk import _native
    L = _native.lib()
    for rows, n, k0, j, k, code in ((21017715, 2076, 496, 4, 248, 5), (23423180, 1131, 339, 3, 339, 2),
                                    (47186238, 768, 12, 3, 3, 4), (52139250, 653, 96, 4, 24, 6),
                                    (28117324, 1242, 104, 4, 104, 6), (50756832, 223, 54, 3, 27, 1),
                                    (5099261, 3822, 3720, 3, 1860, 4), (16484397, 3913, 1752, 3, 438, 5)):
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, rows, n, n, k0, j, k, 0, code, 4096, 4096, buf, 1024) == 0
        for grid, block in re.findall(r"grid=(\d+) block=(\d+)", buf.value.decode()):
            assert int(grid) * int(block) < 1 << 32, buf.value


def test_the_workspace_a_call_uses_stays_within_the_figure_at_its_address():
    # (more calls go through one kernel than that figure tells: it stays what callers have sized buffers by)
    import random
    from approx_topk import _native
    L = _native.lib()
    rng = random.Random(7)
    for _ in range(4000):
        code, j, k_mult = rng.choice((0, 1, 2, 6, 7)), rng.randint(1, 4), rng.choice((2, 3, 4, 8))
        n = int(2 ** rng.uniform(6, 19))
        k = max(1, int(2 ** rng.uniform(2, 13)) // k_mult) * j
        if k * k_mult > n:
            continue
        rows = int(2 ** rng.uniform(0, 14))
        args = (rows, n, n + rng.choice((0, 0, 1, 8)), k * k_mult, j, k, 0, code)
        at = L.atk_topk_workspace_bytes_at(4096, *args)
        used = L.atk_topk_workspace_bytes_used(4096, *args)
        assert used in (0, L.atk_topk_workspace_bytes(rows, n, k * k_mult, j, k, 0, code)) and used <= at, args
        buf = ctypes.create_string_buffer(1024)
        assert L.atk_describe(4096, *args, 4096, 4096, buf, 1024) == 0
        assert (used == 0) == buf.value.startswith(b"fused_"), (args, buf.value)


def _plan(dtype, rows, n, k, j, k_mult=1):
    from approx_topk import _native
    buf = ctypes.create_string_buffer(1024)
    code = _native.dtype_code(dtype)
    assert _native.lib().atk_describe(4096, rows, n, n, k * k_mult, j, k, 0, code, 4096, 4096, buf, 1024) == 0
    text = buf.value.decode()
    found = re.search(r"V=(\d+), W=(\d+), .*? grid=(\d+) .* slabs=(\d+)", text)
    return tuple(int(v) for v in found.groups()) + (text,)


def test_slabs_are_cut_to_one_turn_of_the_cus_where_that_was_measured_faster():
    f32, f16, i8, f64 = torch.float32, torch.float16, torch.int8, torch.float64
    # 16-byte loads in eight waves, and eight-byte elements: no more workgroups than CUs, whatever a slab grows by
    for dtype in (f32, f16, f64):
        for rows in list(range(65, 128, 3)) + [85, 86, 127]:
            vec, waves, grid, slabs, text = _plan(dtype, rows, 1 << 20, 64, 2)
            if slabs > 1 and waves == 8 and (vec > 1 or dtype is f64):
                assert grid <= 256 and grid > 128, text
    assert _plan(f32, 86, 1 << 20, 64, 2)[:4] == (4, 8, 172, 2)
    # four waves: two workgroups a CU stay, where a slab would get more than a third longer; no more than two
    assert _plan(f16, 2, 45395679, 150, 2)[1:3] == (4, 512)
    assert _plan(f16, 4, 1 << 25, 62, 2)[1:3] == (4, 512)
    assert _plan(f16, 3, 1 << 25, 198, 2)[1:3] == (4, 510)
    # (but queues of three and four of 2-byte elements)
    assert _plan(f16, 1, 1 << 26, 4096, 4)[1:3] == (4, 256)
    # one-element loads: two of three slabs stay three
    for dtype in (i8, f16, f32):
        for rows in range(86, 129):
            vec, waves, grid, slabs, text = _plan(dtype, rows, 40001, 240, 1)
            assert vec > 1 or slabs != 2 or waves < 8, text


def test_merges_that_select_are_not_given_more_than_a_workgroup_reads_quickly():
    # one-element loads keep a slab more where one fewer would have the merge select from more than 8192 queues
    assert _plan(torch.bfloat16, 1, 3212725, 24, 1, 8)[::3] == (1, 86)
    assert _plan(torch.float16, 1, 2581297, 24, 1, 8)[::3] == (1, 86)
    # ... and are cut as ever with fewer
    assert _plan(torch.float16, 2, 1319472, 444, 2, 2)[::3] == (1, 18)


def test_slabs_are_raised_to_a_workgroup_a_cu_only_where_that_was_measured_faster():
    f32, f16, bf16 = torch.float32, torch.float16, torch.bfloat16
    assert _plan(f16, 7, 1 << 22, 32, 4, 2)[2:4] == (252, 36) and _plan(f32, 2, 1 << 23, 1024, 4, 4)[2] == 256
    # up to 32 MiB with 16-byte loads: 4-byte elements from 96 workgroups on not, shorter ones by half and more
    assert _plan(f32, 8, 1 << 20, 72, 3, 2)[:4] == (4, 8, 128, 16)
    assert _plan(bf16, 1, 11732747, 16, 1, 2)[3] == _plan(bf16, 1, 11732747, 32, 1)[3] == 179
    assert _plan(f16, 41, 285696, 36, 2, 2)[3] == 6


def test_slabs_of_four_byte_elements_do_not_all_start_in_step():
    # 85 slabs of 2^23 elements are 1.5 KiB off a multiple of 128 KiB
    for dtype in (torch.float32, torch.int32):
        for k in (16, 32, 64, 128, 256, 1024):
            vec, _, grid, _, text = _plan(dtype, 3, 1 << 23, k, 2)
            assert vec > 1 or grid != 255, text
    assert _plan(torch.int32, 3, 1 << 22, 64, 2)[:4] == (1, 8, 255, 85)


# (type, rows, n, k, j, k_mult): calls timed in one kernel and in two, at least 20 % apart: the planner takes the faster one
ONE = [(torch.bfloat16, 4, 32768, 333, 3, 2), (torch.int32, 4, 65536, 433, 1, 2), (torch.int16, 26, 8192, 88, 4, 3),
       (torch.float16, 134, 70338, 1292, 4, 2), (torch.int32, 86, 131072, 878, 2, 4), (torch.float32, 537, 32768, 32, 4, 8),
       (torch.int16, 338, 28275, 300, 4, 2), (torch.float16, 20, 32768, 161, 1, 2)]
TWO = [(torch.int32, 106, 8192, 44, 4, 2), (torch.float16, 617, 56648, 6, 1, 8), (torch.bfloat16, 723, 10369, 20, 4, 4),
       (torch.float16, 3, 158368, 84, 2, 4), (torch.bfloat16, 2, 377089, 36, 1, 2), (torch.bfloat16, 73, 336227, 80, 1, 8)]


@pytest.mark.parametrize("kernels,calls", [("fused_regs_kernel<", ONE), ("stream_kernel<", TWO)], ids=["one", "two"])
def test_one_kernel_or_two_follows_the_faster_plan(kernels, calls):
    from approx_topk import _native
    for dtype, rows, n, k, j, k_mult in calls:
        buf = ctypes.create_string_buffer(1024)
        assert _native.lib().atk_describe(4096, rows, n, n, k * k_mult, j, k, 0, _native.dtype_code(dtype), 4096, 4096, buf, 1024) == 0
        assert buf.value.decode().startswith(kernels), (dtype, rows, n, k, j, k_mult, buf.value)


def test_a_refused_size_leaves_nothing_behind_for_the_next_call():
    # (8.0 and 8 are one key of a dictionary)
    from approx_topk import _native
    x = torch.zeros(3, 64)
    for k in (8.0, 8):
        shape = _native._call_constants(x, k, False, torch.int64)[3]
        assert [type(size) for size in shape] == [int, type(k)]
