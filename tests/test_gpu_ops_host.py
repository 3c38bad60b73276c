"""The torch-tensor calls of ops.py around the kernels: which device and stream they run on, and whose scratch they use."""
import threading

import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _dense_calls(device, seed):
    """Name -> call, on tensors of `device`: one call per format, each of them cut along K through fp32 scratch."""
    from ksanallm_amd import lib as L
    from ksanallm_amd import ops
    g = H.gen(seed)
    m, n, k = 530, 1280, 4096
    for kind in (L.KIND_W4A16, L.KIND_FP8_BLOCKWISE, L.KIND_W4A8):
        d = L.select_tile(kind, m, n, k, H.BF16)
        assert d["kernel"] == 1 and d["split_k"] > 1
    codes = torch.randint(-2**31, 2**31 - 1, (k // 8, n), generator=g, dtype=torch.int32).to(device)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16).to(device)
    s16 = (torch.rand((k // 128, n), generator=g) * 0.01).to(torch.bfloat16).to(device)
    w, s = ops.repack_weight(codes, L.SRC_GPTQ, 1, k, n), ops.repack_scales(s16, L.SCALE_GN, 1, k, n, 128)
    fw = ops.fp8_repack_weight(torch.randint(0, 0x78, (n, k), generator=g, dtype=torch.uint8).to(device))
    fs = (torch.rand((n // 128, k // 128), generator=g) * 1e-3).to(device)
    w8 = ops.w4a8_repack_weight(torch.randint(0, 256, (k, n // 2), generator=g, dtype=torch.uint8).to(device))
    one = torch.tensor([0.05], dtype=torch.float32).to(device)
    s8 = (torch.rand((k // 128, n), generator=g) * 0.01).half().to(device)
    torch.cuda.synchronize(device)
    return {
        "w4a16": lambda: ops.w4a16_gemm(x, w, s, None, n, k, 128),
        "w4a16_f32": lambda: ops.w4a16_gemm_f32(x, w, s, None, n, k, 128),
        "fp8": lambda: ops.fp8_blockwise_gemm(*ops.per_token_group_quant_fp8(x, k), fw, fs),
        "w4a8": lambda: ops.w4a8_gemm(*ops.w4a8_static_quant(x, one), w8, s8, 0.035, n),
    }


def test_threads_on_streams_of_their_own_share_no_scratch():
    """Calls whose partial sums go through scratch, from four threads on four streams at once, give the bits they give alone."""
    calls = [_dense_calls("cuda", 90 + t) for t in range(4)]
    alone = [{name: f().clone() for name, f in c.items()} for c in calls]
    torch.cuda.synchronize()
    failed = []

    def work(t):
        with torch.cuda.stream(torch.cuda.Stream()):
            for turn in range(15):
                for name, f in calls[t].items():
                    y = f()
                    torch.cuda.current_stream().synchronize()
                    if not torch.equal(y, alone[t][name]):
                        failed.append((t, turn, name))
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_tensors_of_another_device_than_the_current_one():
    """A call runs on its tensors' device and that device's stream; the current device stays what it was."""
    calls = _dense_calls("cuda:1", 99)
    with torch.cuda.device(1):
        ref = {name: f().clone() for name, f in calls.items()}
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
    with torch.cuda.device(0):
        prev = torch.cuda.current_stream(1)
        torch.cuda.set_stream(side)   # makes device 1 current as well
        torch.cuda.set_device(0)
        try:
            for name, f in calls.items():
                y = f()
                assert y.device.index == 1 and torch.cuda.current_device() == 0
                side.synchronize()    # the stream the call has to have run on
                assert torch.equal(y, ref[name]), name
        finally:
            torch.cuda.set_stream(prev)
            torch.cuda.set_device(0)
