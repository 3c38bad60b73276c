"""The host side of ops.py's hot calls on a machine without a GPU: what is refused, and before which other step.  A call on CPU
tensors goes through its size checks and the allocation of its outputs and is refused (AssertionError) before any launch."""
import threading
import time

import pytest
import torch


def test_allocation_runs_without_the_interpreter_lock():
    """An allocation that takes its time (here: outputs that torch is told to fill) does not stop the other Python threads: one
    that wakes every millisecond goes on waking.  Under the lock it would wake at most between the call's two allocations and
    around them, however long these take."""
    from ksanallm_amd import ops
    before = torch.are_deterministic_algorithms_enabled(), torch.utils.deterministic.fill_uninitialized_memory, torch.get_num_threads()
    stop, ticks = threading.Event(), []

    def tick():
        while not stop.is_set():
            time.sleep(0.001)
            ticks.append(time.perf_counter())
    thread = threading.Thread(target=tick)
    torch.use_deterministic_algorithms(True)
    torch.utils.deterministic.fill_uninitialized_memory = True
    torch.set_num_threads(1)
    try:
        thread.start()
        time.sleep(0.02)
        t0 = time.perf_counter()
        with pytest.raises(AssertionError, match="device-resident"):
            ops.moe_topk_softmax(torch.zeros((1, 8)), 1 << 26)   # two outputs of 256 MiB
        t1 = time.perf_counter()
    finally:
        stop.set()
        thread.join()
        torch.use_deterministic_algorithms(before[0])
        torch.utils.deterministic.fill_uninitialized_memory = before[1]
        torch.set_num_threads(before[2])
    assert t1 - t0 > 0.02, "the allocation was over too soon to tell (%.3f s)" % (t1 - t0)
    woke = sum(t0 < t < t1 for t in ticks)
    assert woke >= 8, "another thread ran %d times in %.3f s" % (woke, t1 - t0)


def test_out_dtype_is_not_looked_at_where_out_is_given():
    from ksanallm_amd import ops
    m, n, k = 2, 32, 128
    a, a_s = torch.zeros((m, k), dtype=torch.uint8), torch.zeros((1, m))
    out = torch.zeros((m, n), dtype=torch.float16)
    for bad in (None, "half"):
        with pytest.raises(AssertionError, match="device-resident"):
            ops.fp8_blockwise_gemm(a, a_s, torch.zeros((n, k), dtype=torch.uint8), torch.zeros((1, 1)), out_dtype=bad, out=out)
        with pytest.raises(AssertionError, match="device-resident"):
            ops.w4a8_gemm(a, a_s, torch.zeros(n * k // 2, dtype=torch.uint8), torch.zeros((1, n), dtype=torch.float16), 1.0, n,
                          out_dtype=bad, out=out)
        with pytest.raises(TypeError):   # without out it names the type to allocate
            ops.fp8_blockwise_gemm(a, a_s, torch.zeros((n, k), dtype=torch.uint8), torch.zeros((1, 1)), out_dtype=bad)


HUGE = 1 << 60   # a size that a caller states beside its tensors: products with it leave 64 bits


def test_declared_sizes_beyond_64_bits_do_not_pass_for_small_ones():
    """The layout that n, k and the number of experts declare is compared with what the tensors hold as an exact number."""
    from ksanallm_amd import ops
    x, w, s = torch.zeros((16, 128), dtype=torch.float16), torch.zeros(16, dtype=torch.uint8), torch.zeros(16, dtype=torch.float16)
    for n, k in ((16, HUGE), (HUGE, 16), (HUGE, HUGE), (1 << 62, 128), (1 << 63, 128)):
        with pytest.raises((ValueError, OverflowError)):
            ops.w4a16_gemm(x, w, s, None, n, k, 128, out=torch.zeros(1, dtype=torch.float16))
    a, a_s = torch.zeros((16, 128), dtype=torch.uint8), torch.zeros((1, 16))
    with pytest.raises(ValueError):
        ops.w4a8_gemm(a, a_s, w, s, 1.0, HUGE, out=torch.zeros(1, dtype=torch.float16))
    ids, tw = torch.zeros((8, 2), dtype=torch.int32), torch.zeros((8, 2))
    for E, hidden, inter in ((HUGE, 128, 128), (16, HUGE, 128), (16, 128, HUGE), (1 << 32, 1 << 16, 1 << 16)):
        with pytest.raises(ValueError):
            ops.fused_moe_w4a16(x, w, s, w, s, ids, tw, E, hidden, inter, 128)


def test_a_tensor_without_dimensions_has_no_rows():
    from ksanallm_amd import ops
    nil = torch.zeros((), dtype=torch.float16)
    out = torch.zeros((1, 16), dtype=torch.float16)
    w, s = torch.zeros(16 * 128 // 2, dtype=torch.uint8), torch.zeros(16, dtype=torch.float16)
    with pytest.raises(IndexError):
        ops.w4a16_gemm(nil, w, s, None, 16, 128, 128, out=out)
    with pytest.raises(IndexError):
        ops.per_token_group_quant_fp8(nil, 128, q=torch.zeros(0, dtype=torch.uint8), s=torch.zeros(0))
    with pytest.raises(IndexError):
        ops.fp8_blockwise_gemm(torch.zeros((1, 128), dtype=torch.uint8), torch.zeros(1), torch.zeros((), dtype=torch.uint8),
                               torch.zeros(1), out=out)


def test_tensors_that_the_caller_gives_are_checked_against_what_the_call_reads_and_writes():
    """Too small a tensor - outputs and the quantizers' arguments as much as weights - is refused by name, before any launch."""
    from ksanallm_amd import ops
    f16, u8, f32 = torch.float16, torch.uint8, torch.float32
    m, n, k = 16, 32, 256
    x, w, s = torch.zeros((m, k), dtype=f16), torch.zeros(n * k // 2, dtype=u8), torch.zeros((k // 128, n), dtype=f16)
    a, a_s = torch.zeros((m, k), dtype=u8), torch.zeros((k // 128, m))
    b, b_s = torch.zeros((n, k), dtype=u8), torch.zeros((1, k // 128))
    good, short = torch.zeros((m, n), dtype=f16), torch.zeros((m, n - 1), dtype=f16)

    def refused(match, fn, *args, **kw):
        with pytest.raises((ValueError, TypeError), match=match):
            fn(*args, **kw)

    def passes_the_checks(fn, *args, **kw):
        with pytest.raises(AssertionError, match="device-resident"):
            fn(*args, **kw)
    for out, check in ((short, refused), (good, None)):
        for fn, args in ((ops.w4a16_gemm, (x, w, s, None, n, k, 128)), (ops.fp8_blockwise_gemm, (a, a_s, b, b_s)),
                         (ops.w4a8_gemm, (a, a_s, w, s, 1.0, n))):
            passes_the_checks(fn, *args, out=out) if check is None else refused("out", fn, *args, out=out)
    refused("out", ops.w4a16_gemm, x, w, s, None, n, k, 128, out=good.to(torch.bfloat16))     # x is float16
    passes_the_checks(ops.fp8_blockwise_gemm, a, a_s, b, b_s, out=good.float())
    refused("x", ops.per_token_group_quant_fp8, x, 2 * k)
    refused("x", ops.per_token_group_quant_fp8, x, k, fuse_silu_mul=True)                     # reads 2 k columns
    passes_the_checks(ops.per_token_group_quant_fp8, x, k // 2, fuse_silu_mul=True)
    refused("q", ops.per_token_group_quant_fp8, x, k, q=torch.zeros((m, k - 1), dtype=u8))
    refused("s", ops.per_token_group_quant_fp8, x, k, s=torch.zeros((1, m)))
    passes_the_checks(ops.per_token_group_quant_fp8, x, k, q=torch.zeros((m, k), dtype=u8), s=torch.zeros((k // 128, m)))
    for kw, count in (({}, 1), ({"per_channel": True}, k), ({"per_token": True}, m)):
        passes_the_checks(ops.w4a8_static_quant, x, torch.ones(count), **kw)
        refused("scale", ops.w4a8_static_quant, x, torch.ones(count - 1), **kw)
        refused("scale", ops.w4a8_static_quant, x, torch.ones(count, dtype=torch.float64), **kw)
    refused("e_bias", ops.moe_grouped_topk, torch.zeros((m, 8)), 2, e_bias=torch.zeros(7))
    passes_the_checks(ops.moe_grouped_topk, torch.zeros((m, 8)), 2, e_bias=torch.zeros(8))
