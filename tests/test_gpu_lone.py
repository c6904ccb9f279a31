"""Head dim 128, one channel per lane (a head over two waves): forward_qk, forward_ov and the one-launch step at the ends of
their supergroups, tiles, chunks and launches."""
import numpy as np
import pytest
import torch

from adkv_amd import _lib, synth
from adkv_amd.kernel import gemv
from tests.test_gpu_parity import _bf16_case, test_checkpointed_segments, test_forward_qk_and_ov

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 7, 8, 9, 63, 64, 65, 72, 127, 129, 200, 511, 512, 513, 519, 520, 528, 1023, 1024, 1097])
def test_tails_tiles_and_chunks_without_checkpoints(gpu, oracle, T):
    """Tiles of 16 tokens, groups of 64, chunks of 512; rows of odd and even length (weights that are and are not aligned)."""
    test_forward_qk_and_ov(gpu, oracle, 1, 3, T, 128)


@pytest.mark.parametrize("B,H,T,S", [(1, 3, 1300, 1024), (1, 2, 1536, 512), (2, 1, 1100, 520), (3, 5, 129, 64)])
def test_segments_that_end_in_and_between_chunks(gpu, oracle, B, H, T, S):
    """Segments of more than a chunk, of unequal length in one workgroup, and several that are padded to whole quads."""
    test_checkpointed_segments(gpu, oracle, B, H, T, 128, S)


@pytest.mark.parametrize("BH,T", [(1024, 70), (1028, 41), (1536, 41), (1540, 24), (2048, 33), (2052, 24)])
def test_workgroup_sizes(gpu, oracle, BH, T):
    """4, 12 and 16 waves to a workgroup, and just beyond what takes one channel per lane (256 CUs)."""
    test_forward_qk_and_ov(gpu, oracle, BH // 4, 4, T, 128)


@pytest.mark.parametrize("T,S", [(603, 256), (1030, 0)])
def test_the_step_and_the_calls_agree_bit_for_bit(gpu, T, S):
    """Where the softmax between them is the same kernel's, halves and segments are added in the same order."""
    B, H, D = 2, 3, 128
    assert _lib.lib().adkv_decode_step_is_fused(B, H, H, T, D, 4, T // S + 1 if S else 0, S, 0) == 1
    kp, vp = ([t.to(gpu) for t in synth.make_params(H, D, seed=i).astuple()] for i in (3, 4))
    k, v = (f(B, H, T + 1, D, seed=5, dtype=torch.float16).to(gpu) for f in (synth.make_k, synth.make_v))
    q = synth.make_q(B, H, D).to(gpu)
    kw = [dict(ckpt=torch.zeros(B, H, T // S + 1, D, 2, dtype=torch.float16, device=gpu), ckpt_interval=S) if S else {} for _ in "kv"]
    caches = [synth.alloc_cache(B, H, T + 8, D, gpu) for _ in "kv"]
    for c, x, p, o in zip(caches, (k, v), (kp, vp), kw):
        gemv.encode_kv(c, x[:, :, :T].contiguous(), *p, np.exp(-4.0), np.exp(4.0), **o)
    two = [c.clone() for c in caches]
    logits = gemv.forward_qk(q, caches[0], k[:, :, T:], *kp, T, np.exp(-4.0), np.exp(4.0), **kw[0])
    w = gemv.softmax_scale_mask(logits, D ** -0.5)
    out = gemv.forward_ov(w, caches[1], v[:, :, T:], *vp, np.exp(-4.0), np.exp(4.0), **kw[1])
    out2, w2 = gemv.decode_step(q, *two, k[:, :, T:], v[:, :, T:], kp, vp, T, D ** -0.5, k_ckpt=kw[0].get("ckpt"),
                                v_ckpt=kw[1].get("ckpt"), ckpt_interval=S)
    torch.cuda.synchronize()
    assert torch.equal(w.contiguous().view(torch.int16), w2.contiguous().view(torch.int16))
    assert torch.equal(out.view(torch.int16), out2.view(torch.int16))
    assert torch.equal(caches[0], two[0]) and torch.equal(caches[1], two[1])


@pytest.mark.parametrize("B,H,T", [(2, 4, 1600), (3, 5, 1541), (65, 4, 520)])
def test_bfloat16_results_of_rows_in_one_piece(gpu, B, H, T):
    """Steps that are neither one launch nor two, without checkpoints: forward_ov's waves write the results themselves."""
    L = _lib.lib()
    assert L.adkv_decode_step_launches(B, H, H, T, 128, 4, 0, 0, 0) == 3
    assert L.adkv_decode_ov_kernel_name(B, H, H, T, 128, 4, 0, 0).startswith(b"lone_kernel")
    _bf16_case(gpu, B, H, H, T, 0, 4)
