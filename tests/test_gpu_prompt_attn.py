"""The prompt attention kernel (rotary, cache writes, attention) against PyTorch in fp64.

Bounds: q and k are rounded to fp16 once after the rotary (2^-11 of each), which moves a score of size s by up to
2^-10 |s|; with |s| of a few units the softmax weights move by under 2^-8, and the fp16 output rounds by 2^-11.
The caches equal the rounded rotary exactly."""

import math

import pytest
import torch

from eptq_amd.kernels import _lib
from eptq_amd.llama import _rope

pytestmark = pytest.mark.gpu


def _run(B, T, H, Hk, L, p0, seed, scale=1.0, back=False):
    g = torch.Generator(device="cuda").manual_seed(seed)
    D = 128
    qkv = (torch.randn((B * T, (H + 2 * Hk) * D), generator=g, device="cuda") * scale).half()
    kc = torch.randn((B, Hk, L, D), generator=g, device="cuda").half()      # rows below p0: an earlier prompt
    vc = torch.randn((B, Hk, L, D), generator=g, device="cuda").half()
    ang = torch.outer(torch.arange(L, device="cuda").float(),
                      1.0 / (10000.0 ** (torch.arange(0, D, 2, device="cuda").float() / D)))
    cos, sin = torch.cat((ang, ang), -1).cos().contiguous(), torch.cat((ang, ang), -1).sin().contiguous()
    pos = torch.arange(p0, p0 + T, device="cuda")
    if back:
        pos = pos.flip(0).contiguous()
    q, k, v = (t.reshape(B, T, -1, D).transpose(1, 2) for t in qkv.split([H * D, Hk * D, Hk * D], dim=-1))
    c, s = cos[pos][None, None], sin[pos][None, None]
    q16, k16 = _rope(q, c, s), _rope(k, c, s)
    k0, v0 = kc.clone(), vc.clone()
    k0.index_copy_(2, pos, k16)
    v0.index_copy_(2, pos, v)
    out = torch.full((B * T, H * D), float("nan"), dtype=torch.float16, device="cuda")
    rc = _lib.load().eptq_llama_prompt_attn(qkv.data_ptr(), pos.data_ptr(), cos.data_ptr(), sin.data_ptr(),
                                            kc.data_ptr(), vc.data_ptr(), out.data_ptr(), B, T, H, Hk, D, L,
                                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(kc, k0) and torch.equal(vc, v0)
    allowed = torch.arange(L, device="cuda")[None, :] <= pos[:, None]
    sc = torch.matmul(q16.double(), k0.double().repeat_interleave(H // Hk, 1).transpose(-1, -2).contiguous()) / math.sqrt(D)
    w = torch.softmax(sc.masked_fill(~allowed, float("-inf")), -1)
    ref = torch.matmul(w, v0.double().repeat_interleave(H // Hk, 1).contiguous()).transpose(1, 2).reshape(B * T, H * D)
    return out, ref


# Token counts around the 16 of a wave and the 64 of a workgroup, cache lengths around the block of 64 rows, a cache
# with earlier rows, grouped heads, large scores (one-hot softmax) and tiny ones (uniform).
@pytest.mark.parametrize("B,T,H,Hk,L,p0,scale,back", [
    (1, 1, 1, 1, 1, 0, 1.0, False),
    (1, 1, 4, 4, 130, 129, 1.0, False),
    (2, 15, 4, 2, 64, 49, 1.0, False),
    (1, 64, 2, 2, 65, 1, 1.0, False),
    (3, 65, 8, 1, 200, 63, 1.0, False),
    (1, 127, 2, 2, 128, 0, 4.0, False),
    (2, 300, 4, 4, 1000, 500, 0.05, False),
    (1, 80, 2, 1, 96, 10, 1.0, True),
])
def test_prompt_attention(B, T, H, Hk, L, p0, scale, back):
    print(f"prompt attention B={B} T={T} H={H}/{Hk} L={L} p0={p0}", flush=True)
    out, ref = _run(B, T, H, Hk, L, p0, T + L, scale, back)
    err = float((out.double() - ref).norm() / ref.norm())
    assert err <= 2.0 ** -11, err     # the same fp16 q, k, v in fp64: only the sums and the output round


def test_prompt_attention_rejects_other_head_dims():
    x = torch.zeros(64, dtype=torch.float16, device="cuda")
    rc = _lib.load().eptq_llama_prompt_attn(*([x.data_ptr()] * 7), 1, 1, 1, 1, 64, 1, 0)
    assert rc == 2


def test_prompt_kernels_only_for_the_caches_batch_and_length():
    """The kernel addresses the caches by sequence: other batches keep the refusal of the PyTorch operators, and a
    prompt longer than the cache and a model with trainable parameters never reach it."""
    from eptq_amd.llama import LlamaConfig, build_synthetic
    model = build_synthetic(LlamaConfig(hidden=256, ffn=256, layers=1, heads=2, kv_heads=2, vocab=64), device="cuda", seed=3)
    model.alloc_cache(1, 8, "cuda")

    def taken(B, T):
        ids = torch.zeros((B, T), dtype=torch.int64, device="cuda")
        return model._hip_prompt(model.embed_tokens(ids), ids, torch.arange(T, device="cuda"))

    assert taken(1, 1) and taken(1, 8)
    assert not taken(1, 9) and not taken(2, 8)
    model.norm.weight.requires_grad_(True)
    assert not taken(1, 8)
    with torch.no_grad():
        assert taken(1, 8)
        with pytest.raises((RuntimeError, IndexError)):
            model.forward_tokens(torch.zeros((2, 4), dtype=torch.int64, device="cuda"), torch.arange(4, device="cuda"))
