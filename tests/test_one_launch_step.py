"""adkv_decode_step where it is one launch: what the measurement hook does to it, and what the library
says about it."""
import ctypes

import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv

D = 128


def _step(gpu, B, H, T, S, workspace):
    kp, vp = (tuple(t.to(gpu) for t in synth.make_params(H, D, seed=3 + i).astuple()) for i in range(2))
    k, v = (f(B, H, T + 1, D, seed=5, dtype=torch.float16, device=gpu) for f in (synth.make_k, synth.make_v))
    q = synth.make_q(B, H, D, seed=6, device=gpu)
    caches = [synth.alloc_cache(B, H, T + 8, D, gpu) for _ in range(2)]
    cks = [torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    states = [torch.zeros(B, H, D, 2, dtype=torch.float16, device=gpu) for _ in range(2)]
    gemv.append_kv_pair(*caches, k[:, :, :T].contiguous(), v[:, :, :T].contiguous(), kp, vp, 0, *states, k_ckpt=cks[0],
                        v_ckpt=cks[1], ckpt_interval=S)
    out, w = gemv.decode_step(q, *caches, k[:, :, T:].contiguous(), v[:, :, T:].contiguous(), kp, vp, T, D ** -0.5,
                              k_ckpt=cks[0], v_ckpt=cks[1], ckpt_interval=S, workspace=workspace)
    torch.cuda.synchronize()
    return [out, w.contiguous(), *caches, *cks]


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,T", [(1, 4, 603), (2, 3, 64), (1, 2, 1000)])
def test_stage_events_do_not_change_what_runs(gpu, B, H, T):
    """A one-launch step keeps its logits and weights out of the workspace, the separate launches do not:
    with the events set the workspace stays untouched and every bit of the result is the same."""
    S = 256
    need = gemv.decode_step_workspace_bytes(B, H, H, T, D, T // S + 1, S)
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=gpu)
    plain = _step(gpu, B, H, T, S, ws)
    assert bool((ws == 0xA5).all())
    events = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
    for e in events:
        e.record()
    _lib.lib().adkv_set_stage_events((ctypes.c_void_p * 4)(*[e.cuda_event for e in events]))
    try:
        timed = _step(gpu, B, H, T, S, ws)
    finally:
        _lib.lib().adkv_set_stage_events(None)
    assert bool((ws == 0xA5).all())
    for a, b in zip(plain, timed):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert events[0].elapsed_time(events[1]) > 0 and events[0].elapsed_time(events[3]) >= events[0].elapsed_time(events[1])


def test_library_says_which_steps_are_one_launch():
    """Without a GPU: the rule of the sizes (256 CUs), masked or not, and the knobs that turn it off."""
    L = _lib.lib()
    fused = lambda B, Hq, H, T, S=256, D=D, bits=4, masked=0: L.adkv_decode_step_is_fused(
        B, Hq, H, T, D, bits, T // S + 1 if S else 0, S, masked)
    for masked in (0, 1):
        assert fused(1, 32, 32, 603, masked=masked) == 1
        assert fused(8, 32, 32, 1000, masked=masked) == 1
        assert fused(1, 32, 32, 1535, 0, masked=masked) == 1
        assert fused(1, 32, 32, 0, masked=masked) == 1
        assert fused(9, 32, 32, 600, masked=masked) == 0          # more heads than CUs
        assert fused(1, 32, 32, 1536, 0, masked=masked) == 0      # a row too long
        assert fused(1, 32, 8, 600, masked=masked) == 0           # grouped queries
        assert fused(1, 32, 32, 600, bits=2, masked=masked) == 0
        assert fused(1, 8, 8, 600, D=256, masked=masked) == 0
        assert fused(128, 32, 32, 4096, masked=masked) == 0       # the other kind, not asked for
    for kernel in (0, 1, 2, 3, 4):
        L.adkv_set_mha_kernel(kernel)
        try:
            assert fused(1, 32, 32, 603) == 0
        finally:
            L.adkv_set_mha_kernel(-1)
    L.adkv_set_fused_step(1)
    try:
        assert fused(128, 32, 32, 4096) == 1 and fused(128, 32, 32, 4096, masked=1) == 0 and fused(1, 32, 32, 603) == 1
    finally:
        L.adkv_set_fused_step(0)


def test_library_says_in_how_many_launches_a_step_runs():
    """Without a GPU, and what the benchmark calls the kernels of such a step."""
    import bench
    L = _lib.lib()
    launches = lambda B, Hq, H, T, S=256, D=D, bits=4, masked=0: L.adkv_decode_step_launches(
        B, Hq, H, T, D, bits, T // S + 1 if S else 0, S, masked)
    names = lambda B, Hq, H, T, D=D, bits=4, S=256: bench.step_kernels(L, B, Hq, H, T, D, bits, T // S + 1, S)
    for masked in (0, 1):
        assert launches(1, 32, 32, 603, masked=masked) == 1
        for n, sizes in ((2, (8, 32, 8, 16001)), (2, (4, 32, 32, 8000)), (2, (64, 32, 32, 663)), (2, (1, 64, 8, 300)),
                         (3, (128, 32, 32, 4096)), (3, (16, 32, 8, 131072)), (3, (1, 64, 8, 300, 0)), (3, (2, 3, 3, 4000, 64))):
            assert launches(*sizes, masked=masked) == n, sizes
        assert launches(4, 8, 8, 8190, D=256, masked=masked) == 2 and launches(2, 8, 2, 5000, bits=2, masked=masked) == 2
    # a table per head pays: its forward_ov adds two or four segments in the workgroup, or does not; half of the CUs
    for n, sizes in ((3, (128, 32, 32, 300)), (3, (64, 32, 32, 1024)), (3, (40, 40, 40, 1000)), (2, (40, 32, 32, 1100)),
                     (2, (64, 40, 40, 600)), (2, (32, 32, 32, 2048)), (2, (8, 32, 32, 8000)), (2, (128, 32, 32, 256)),
                     (2, (128, 32, 32, 150, 128)), (2, (128, 32, 32, 250, 128)), (3, (128, 32, 32, 500, 128)), (3, (16, 32, 32, 8000, 128)), (3, (100, 32, 32, 1000, 512)),
                     (2, (32, 32, 32, 4000, 512)), (2, (64, 32, 32, 1500, 512))):
        assert launches(*sizes) == n, sizes
    for bad in ((2, 6, 4, 100), (2, 6, 2, 100), (0, 8, 8, 100), (1, 8, 8, -1)):
        assert launches(*bad) == 3
    assert launches(2, 16, 8, 100, D=256) == 3 and launches(1, 8, 8, 100, bits=3) == 3
    assert names(1, 32, 32, 603) == ("small_step_kernel",)
    assert names(8, 32, 8, 16001) == ("step_segments_kernel", "step_combine_kernel")
    assert names(128, 32, 32, 4096)[0].startswith("qk_ft_kernel (") and len(names(128, 32, 32, 4096)) == 3
    L.adkv_set_mha_kernel(0)
    try:
        assert launches(8, 32, 8, 16001) == 3
    finally:
        L.adkv_set_mha_kernel(-1)


def test_library_and_benchmark_name_the_first_kernel_of_a_step():
    """Without a GPU (256 CUs): one channel per lane up to 12 waves of 64 channels per CU (wide heads 16, eight query heads 8),
    the other kernel beyond, longer segments and in one launch."""
    import bench
    L = _lib.lib()

    def name(B, Hq, H, T, D=D, bits=4, S=256, masked=0):
        n = T // S + 1 if S else 0
        first = L.adkv_decode_step_kernel_name(B, Hq, H, T, D, bits, n, S, masked)
        if not masked and L.adkv_decode_step_launches(B, Hq, H, T, D, bits, n, S, 0) < 3:
            assert bench.step_kernels(L, B, Hq, H, T, D, bits, n, S)[0] == first.decode()
        return first.decode() if first else None

    lone = "step_lone_kernel, %d-wave workgroups"
    for bits in (4, 2):
        for waves, sizes in ((4, (4, 32, 32, 2048)), (12, (6, 32, 32, 2048)), (0, (7, 32, 32, 2048)), (4, (4, 32, 16, 2048)),
                             (8, (8, 32, 16, 2048)), (12, (12, 32, 16, 2048)), (0, (13, 32, 16, 2048)), (4, (8, 32, 8, 2048)),
                             (8, (16, 32, 8, 2048)), (12, (24, 32, 8, 2048)), (0, (25, 32, 8, 2048)), (4, (8, 64, 8, 2048)),
                             (8, (16, 64, 8, 2048)), (0, (17, 64, 8, 2048))):
            assert name(*sizes, bits=bits) == name(*sizes, bits=bits, masked=1) == (lone % waves if waves else "step_segments_kernel")
    for waves, sizes in ((4, (4, 16, 16, 2048, 256)), (12, (6, 16, 16, 2048, 256)), (16, (8, 16, 16, 2048, 256)),
                         (0, (9, 16, 16, 2048, 256)), (8, (4, 8, 8, 2048, 512)), (16, (8, 8, 8, 2048, 512)), (0, (9, 8, 8, 2048, 512))):
        assert name(*sizes) == (lone % waves if waves else "step_segments_kernel"), sizes
    assert name(2, 8, 2, 1500, S=512) == "step_segments_kernel"               # segments beyond 256 tokens
    assert name(1, 32, 32, 603) == name(1, 32, 32, 603, masked=1) == "small_step_kernel"
    assert name(128, 32, 32, 4096) is None and name(1, 6, 4, 100) is None
    L.adkv_set_fused_step(1)
    try:
        assert name(128, 32, 32, 4096) == "decode_ft_kernel" and name(128, 32, 32, 4096, masked=1) is None
    finally:
        L.adkv_set_fused_step(0)


def test_library_says_whether_the_values_have_waves_beside_the_keys():
    """Without a GPU (256 CUs): 24 units held with up to four waves of keys per CU, 16 up to eight, none beyond and in the other
    kernels.  The rows of test_gpu_step_beside.test_most_waves, then what lies behind them."""
    L = _lib.lib()
    ahead = lambda B, Hq, H, D, T, bits, S=256: L.adkv_decode_step_values_ahead(B, Hq, H, T, D, bits, T // S + 1 if S else 0, S)
    for n, rows in ((24, ((2, 32, 32, 128, 2000, 4), (4, 32, 16, 128, 2048, 4), (8, 64, 8, 128, 2000, 4), (2, 32, 32, 128, 1999, 2),
                          (2, 16, 16, 256, 2000, 4))),
                    (16, ((2, 32, 32, 128, 2100, 4), (4, 32, 16, 128, 2049, 4), (2, 16, 16, 256, 2064, 4), (4, 32, 32, 128, 2047, 4),
                          (4, 32, 32, 128, 1800, 2), (8, 32, 16, 128, 2048, 4), (5, 32, 8, 128, 6400, 4), (5, 64, 8, 128, 5633, 4),
                          (4, 16, 16, 256, 2040, 4), (3, 8, 8, 512, 2500, 4), (1, 8, 8, 512, 8192, 4), (1, 8, 8, 512, 300, 4))),
                    (0, ((4, 32, 32, 128, 2049, 4), (8, 32, 16, 128, 2049, 4), (16, 64, 8, 128, 2049, 4), (4, 16, 16, 256, 2049, 4),
                         (2, 8, 8, 512, 4097, 4), (8, 32, 8, 128, 16001, 4), (1, 32, 32, 128, 603, 4), (128, 32, 32, 128, 4096, 4)))):
        for row in rows:
            assert ahead(*row) == n, row
    assert ahead(2, 8, 2, 128, 1500, 4, 512) == 0                              # segments beyond 256 tokens
    for bad in ((0, 8, 8, 128, 100, 4), (1, 6, 4, 128, 100, 4), (1, 8, 8, 128, -1, 4), (1, 8, 8, 128, 100, 3), (2, 16, 8, 256, 100, 4)):
        assert ahead(*bad) == 0
    L.adkv_set_mha_kernel(0)
    try:
        assert ahead(2, 32, 32, 128, 2000, 4) == 0
    finally:
        L.adkv_set_mha_kernel(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("H,T,S", [(4, 200, 64), (3, 600, 256)])
def test_one_launch_step_replays_from_a_captured_graph(gpu, H, T, S):
    from tests.test_gpu_parity import test_decode_step_replays_from_a_captured_graph as replays
    assert _lib.lib().adkv_decode_step_is_fused(2, H, H, T, D, 4, (T + 8) // S + 1, S, 0) == 1
    replays(gpu, H, H, T, S, 4)
