"""The host side of ops.py's hot calls on a machine without a GPU: what is refused, and before which other step.  A call on CPU
tensors goes through its size checks and the allocation of its outputs and is refused (AssertionError) before any launch."""
import threading
import time

import pytest
import torch


def test_allocation_runs_without_the_interpreter_lock():
    """An allocation that takes its time (here: outputs that torch is told to fill) does not stop the other Python threads."""
    from ksanallm_amd import ops
    before = torch.are_deterministic_algorithms_enabled(), torch.utils.deterministic.fill_uninitialized_memory, torch.get_num_threads()
    stop, gaps = threading.Event(), []

    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.001)
            now = time.perf_counter()
            gaps.append(now - last)
            last = now
    thread = threading.Thread(target=tick)
    torch.use_deterministic_algorithms(True)
    torch.utils.deterministic.fill_uninitialized_memory = True
    torch.set_num_threads(1)
    try:
        thread.start()
        time.sleep(0.02)
        del gaps[:]
        t0 = time.perf_counter()
        with pytest.raises(AssertionError, match="device-resident"):
            ops.moe_topk_softmax(torch.zeros((1, 8)), 1 << 28)   # two outputs of 1 GiB
        took = time.perf_counter() - t0
    finally:
        stop.set()
        thread.join()
        torch.use_deterministic_algorithms(before[0])
        torch.utils.deterministic.fill_uninitialized_memory = before[1]
        torch.set_num_threads(before[2])
    assert took > 0.05, "the allocation was over too soon to tell (%.3f s)" % took
    assert max(gaps) < took / 3, "another thread stood still for %.3f of %.3f s" % (max(gaps), took)


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
