"""The Hugging Face TurboQuant cache on the GPU, end to end on a tiny random
Llama (head_dim 128, GQA 2:1, two layers), teacher-forced: prompt, then one
token per step.

The oracle is the reference's cache restated on the CPU
(oracle/turboquant_cache.py) driving the same model on the CPU with eager
attention.  The scenario spills exactly once (prompt of 40 tokens, residual
of 64, 30 decode steps), so the reference's re-quantisation of older tokens
at later spills does not arise and both caches hold the same codes.

Logits of every step agree within |gpu - oracle| <= 2e-2 + 2e-2 |oracle|:
the attention outputs themselves meet 2e-3 + 1e-2 |ref| (the paged decode
bar), propagated through two layers and the output projection.
"""
import copy

import pytest
import torch
from transformers import LlamaConfig, LlamaForCausalLM

from oracle import turboquant as TQ
from oracle.turboquant_cache import OracleTurboQuantCache
from vramancer_amd.turboquant_cache import TurboQuantCache, enable_paged_attention

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _say(msg):
    print(f"[case] {msg}", flush=True)


def _model():
    cfg = LlamaConfig(vocab_size=256, hidden_size=512, intermediate_size=256, num_hidden_layers=2,
                      num_attention_heads=4, num_key_value_heads=2, head_dim=128, max_position_embeddings=512)
    cfg._attn_implementation = "eager"
    torch.manual_seed(0)
    return LlamaForCausalLM(cfg).eval()


@torch.no_grad()
def _run(model, cache, ids, steps):
    out = [model(ids[:, :-steps], past_key_values=cache, use_cache=True).logits[:, -1].float().cpu()]
    for i in range(steps, 0, -1):
        pos = ids.shape[1] - i
        out.append(model(ids[:, pos:pos + 1], past_key_values=cache, use_cache=True).logits[:, -1].float().cpu())
    return torch.stack(out, 1)


def _close(got, want, what):
    err = (got - want).abs()
    bad = err > 2e-2 + 2e-2 * want.abs()
    assert not bad.any(), f"{what}: {int(bad.sum())} logits off, max err {err.max():.3e}"


@pytest.fixture(scope="module")
def setting():
    model = _model()
    ids = torch.randint(0, 256, (2, 70), generator=torch.Generator().manual_seed(3))
    oracle = OracleTurboQuantCache(2, TQ.make_params(128, 3, seed=11), residual_length=64)
    ref = _run(model, oracle, ids, 30)
    assert oracle.layers[0].spills == 1
    return model, ids, ref


@pytest.mark.parametrize("paged", [True, False], ids=["paged-decode", "materialised"])
def test_turboquant_cache_matches_reference_cache(setting, paged):
    model, ids, ref = setting
    _say(f"hf cache paged={paged}")
    gpu_model = copy.deepcopy(model).to(DEV)
    if paged:
        enable_paged_attention(gpu_model)
    else:
        gpu_model.set_attn_implementation("sdpa")
    torch.manual_seed(11)  # the compressor draws its rotation as the reference's does
    cache = TurboQuantCache(2, 128, bits_per_angle=3, residual_length=64, device=DEV, paged_attention=paged)
    got = _run(gpu_model, cache, ids.to(DEV), 30)
    assert cache.get_seq_length() == 70
    layer = cache.layers[1]
    assert (layer._n_comp, layer._res_len) == (64, 6)
    _close(got, ref, f"paged={paged}")


def test_turboquant_cache_decode_attention_matches_materialised(setting):
    """The paged decode step (TurboQuant pages + residual merged by
    log-sum-exp) against SDPA over the same cache's materialised keys/values."""
    model, ids, _ = setting
    _say("paged step vs materialised")
    torch.manual_seed(11)
    cache = TurboQuantCache(2, 128, bits_per_angle=3, residual_length=32, device=DEV, paged_attention=True)
    layer = cache.layers[0]
    g = torch.Generator().manual_seed(4)
    # prompt, then steps that spill and refill the residual; the 60-token update grows the
    # residual pool while it holds a token (copy, new page / slot table), the next one spills it
    for s in (40, 1, 1, 30, 1, 60, 1):
        k = torch.randn(2, 2, s, 128, generator=g).to(DEV)
        layer.update(k, torch.randn(2, 2, s, 128, generator=g).to(DEV))
        q = torch.randn(2, 4, 1, 128, generator=g).to(DEV)
        got = layer.attend_decode(q, 0.08)[:, 0].float().cpu()
        K, V = layer.materialize()
        Kr = K.float().cpu().repeat_interleave(2, dim=1)
        Vr = V.float().cpu().repeat_interleave(2, dim=1)
        w = torch.softmax(0.08 * (Kr @ q.float().cpu()[:, :, 0, :, None])[..., 0], -1)
        want = (w[..., None] * Vr).sum(2)
        err = (got - want).abs()
        assert (err <= 2e-3 + 1e-2 * want.abs()).all(), f"step {s}: max err {err.max():.3e} view {layer._view}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim,bits,B,n_c,n_r", [
    (64, 4, 4, 2000, 101),   # many partials of the pages, several of the residual
    (64, 4, 1, 16, 1),       # one partial of each
    (128, 3, 3, 160, 160),   # as many pages in both passes: their workspaces stay apart
    (96, 2, 2, 3000, 33),
    (256, 5, 2, 48, 17),     # head_dim above 128, generic pages
])
def test_merged_step_matches_two_decodes(dtype, head_dim, bits, B, n_c, n_r):
    """The one merge of both passes' partials against the two decodes combined
    by log-sum-exp.  The passes are the same, so float32 outputs differ by the
    order of the sum over at most 600 partials of weight sum 1 (600 x 2^-24 of
    the largest value) and by the rounding of the two log-sum-exps (|lse| < 16:
    2^-20 of a value each), together below 4e-5 for |v| < 1 here; the 16-bit
    outputs by one more rounding of theirs (2^-11, 2^-8 relative)."""
    from vramancer_amd import tq_pages
    from vramancer_amd.paged_attention_cuda import combine_attention, paged_attention_decode

    _say(f"merged step {dtype} d{head_dim} b{bits} B{B} {n_c}+{n_r}")
    torch.manual_seed(5)
    cache = TurboQuantCache(1, head_dim, bits_per_angle=bits, residual_length=n_r, device=DEV, paged_attention=True)
    layer = cache.layers[0]
    g = torch.Generator().manual_seed(6)
    for s in (n_c, n_r):
        k = torch.randn(B, 2, s, head_dim, generator=g).to(DEV, dtype)
        layer.update(k, (torch.rand(B, 2, s, head_dim, generator=g) - 0.5).to(DEV, dtype))
    assert layer._view == (n_c, n_r)
    q = torch.randn(B, 6, 1, head_dim, generator=g).to(DEV, dtype)
    got = layer.attend_decode(q, 0.09)
    assert got.dtype == dtype and tuple(got.shape) == (B, 1, 6, head_dim)
    pj, pr = -(-n_c // 16), -(-n_r // 16)
    q3 = q[:, :, 0].float().contiguous()
    l1, l2 = (torch.empty((B, 6), device=DEV) for _ in range(2))
    o1 = tq_pages.paged_attention_decode_turbo(q3, layer._tq_pool, layer._table("tq", pj), layer._lengths(n_c), 0,
                                               layer.compressor, scale=0.09, lse=l1, qjl=False)
    o2 = paged_attention_decode(q3, layer._res_pool, layer._table("res", pr), layer._lengths(n_r), 0, scale=0.09,
                                lse=l2)
    want = combine_attention(o1, l1, o2, l2)
    rel = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    err = (got[:, 0].float() - want).abs()
    assert (err <= 4e-5 + rel * want.abs()).all(), f"max err {err.max():.3e}"
