"""The TurboQuant kernels with 16 rows per wavefront on the GPU.

Encoder:

Calls of 2048 rows and more take it; the same rows in smaller calls take one
row per wavefront, the path the oracle tests hold to the reference.  Both give
the same codes bit for bit, whatever the rows hold: values at sector edges
(zero, constant, one-hot and sparse rows, whose angles are exact multiples of
pi / 4), magnitudes down to the denormals and up to overflow, infinities and
NaN (a NaN norm stays NaN; its payload is not pinned).
"""
import math

import pytest
import torch

from oracle import turboquant as TQ
from test_gpu_turboquant import _student_t
from vramancer_amd import tq_pages
from vramancer_amd.kv_quantizer import KVCacheCompressor, _pack_bits, _pack_values

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _say(msg):
    print(f"[case] {msg}", flush=True)


def _rows(n, d, dtype, seed):
    x = _student_t(n, d, seed).float()
    at = 37
    for row in (torch.zeros(d), -torch.zeros(d), torch.ones(d), torch.eye(d)[d // 2] * 3, torch.full((d,), math.inf),
                torch.full((d,), 6e4), x[1] * 1e-20, x[2] * 1e-38, x[3] * 1e-44, x[4] * 1e19, x[5] * 1e36):
        x[at] = row
        at += 5
    x[at, 3] = math.nan
    x[at + 1, ::2] = 0
    x[at + 2, 1:] = 0
    return x.to(dtype)


def _bits16(t):
    """fp16 bits, every NaN alike."""
    t = t.reshape(-1).cpu()
    return torch.where(t.isnan(), torch.full_like(t, math.nan), t).view(torch.int16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("head_dim,bits", [(128, 2), (128, 3), (128, 4), (96, 3), (70, 4), (64, 2), (64, 3), (64, 4),
                                           (33, 3)])
def test_tile_codes_equal_row_codes(head_dim, bits, dtype):
    _say(f"tile codes {head_dim} {bits} {dtype}")
    torch.manual_seed(head_dim + bits)
    comp = KVCacheCompressor(head_dim, bits).to(DEV)
    n = 2048 + 13  # the last wavefront has 13 rows
    x = _rows(n, head_dim, dtype, bits).to(DEV)
    shifted = torch.empty(n * head_dim + 1, dtype=dtype, device=DEV)[1:].reshape(n, head_dim).copy_(x)
    for rows in (x, shifted):  # 16-byte aligned rows, and rows off every alignment
        raw = comp.compress(rows, pack=False)
        parts = [comp.compress(rows[s:s + 1024], pack=False) for s in range(0, n, 1024)]
        for key in ("radius", "qjl_norms"):
            assert torch.equal(_bits16(raw[key]), _bits16(torch.cat([p[key] for p in parts]))), key
        assert torch.equal(torch.cat(raw["angles"], -1), torch.cat([torch.cat(p["angles"], -1) for p in parts]))
        assert torch.equal(raw["qjl_signs"], torch.cat([p["qjl_signs"] for p in parts]))
    for m in (1, 17, n):  # packed in the same launch, at any row count
        packed = comp.compress(x[:m])
        assert torch.equal(packed["angles_packed"], _pack_values(torch.cat(raw["angles"], -1)[:m], bits))
        assert torch.equal(packed["qjl_signs_packed"], _pack_bits(raw["qjl_signs"][:m]))
        assert torch.equal(_bits16(packed["radius"]), _bits16(raw["radius"][:m]))
        assert torch.equal(_bits16(packed["qjl_norms"]), _bits16(raw["qjl_norms"][:m]))


@pytest.mark.parametrize("head_dim,bits", [(128, 3), (128, 4), (80, 2), (64, 2), (64, 3), (48, 4)])
def test_tile_pages_equal_small_writes(head_dim, bits):
    """Pages written in one call (2 x 2304 rows) equal page-by-page writes,
    with partly filled pages, an empty one and ids outside the pool."""
    _say(f"tile pages {head_dim} {bits}")
    torch.manual_seed(head_dim)
    comp = KVCacheCompressor(head_dim, bits).to(DEV)
    P, L, KH, NP = 40, 2, 4, 36
    g = torch.Generator().manual_seed(bits)
    k, v = (_rows(NP * KH * 16, head_dim, torch.bfloat16, s).reshape(NP, KH, 16, head_dim).to(DEV) for s in (1, 2))
    k[k.isnan()] = 0.0  # pages compare as bytes, which leaves NaN payloads out
    v[v.isnan()] = 0.0
    k, v = k.clamp(-1e18, 1e18), v.clamp(-1e18, 1e18)
    ids = torch.randperm(P, generator=g)[:NP].to(torch.int32)
    ids[5], ids[9] = -1, P
    n_valid = torch.randint(1, 17, (NP,), generator=g).to(torch.int32)
    n_valid[3], n_valid[4] = 0, 16
    ids, n_valid = ids.to(DEV), n_valid.to(DEV)
    a = tq_pages.allocate_pool(P, L, KH, comp, DEV)
    b = tq_pages.allocate_pool(P, L, KH, comp, DEV)
    a.fill_(7)
    b.fill_(7)
    tq_pages.quantize_pages(a, 1, ids, k, v, comp, n_valid)
    for n in range(NP):
        tq_pages.quantize_pages(b, 1, ids[n:n + 1], k[n:n + 1].contiguous(), v[n:n + 1].contiguous(), comp,
                                n_valid[n:n + 1])
    assert torch.equal(a.cpu(), b.cpu())
    # and the codes are the codec's
    got = tq_pages.read_pages(a, 1, ids[4:5], comp)
    ref = comp.compress(torch.stack([k[4], v[4]]), pack=False)
    assert torch.equal(got["angles"].reshape(-1, got["angles"].shape[-1]).cpu(), torch.cat(ref["angles"], -1).cpu())
    assert torch.equal(got["qjl_signs"][0, 0].reshape(KH * 16, -1).cpu(), ref["qjl_signs"][:KH * 16].cpu())


@pytest.mark.parametrize("head_dim,bits", [(128, 2), (128, 3), (128, 4), (96, 3), (70, 4), (64, 2), (64, 3), (64, 4),
                                           (33, 3)])
def test_tile_decompress_matches_oracle(head_dim, bits):
    """Decompression of raw and packed codes is the oracle's, bit for bit (zeros
    and NaN apart), over radii of every kind; 16,384 rows and more of raw codes
    at padded dim 128 take the tiles, packed codes at any count."""
    _say(f"tile decompress {head_dim} {bits}")
    p = TQ.make_params(head_dim, bits, seed=head_dim)
    torch.manual_seed(head_dim)
    comp = KVCacheCompressor(head_dim, bits).to(DEV)
    pd = comp._padded_dim
    n = 16384 + 5
    g = torch.Generator().manual_seed(bits)
    radius = (torch.rand(n, generator=g) * 20).half()
    radius[::97] = torch.tensor([0.0, -0.0, math.inf, math.nan, 6e-8, 65504.0, -3.0]).half().repeat(n)[:radius[::97].numel()]
    bins = torch.randint(0, 1 << bits, (n, pd - 1), generator=g, dtype=torch.uint8)
    dims = [pd >> (l + 1) for l in range(comp._n_levels)]
    raw = {"radius": radius, "angles": list(torch.split(bins, dims, -1)), "qjl_signs": torch.zeros(n, pd // 2, dtype=torch.uint8),
           "qjl_norms": torch.zeros(n, 1).half(), "shape": (n, head_dim)}
    want = TQ.decompress(p, dict(raw, radius=radius[:, None])).reshape(n, head_dim)
    dev = {k: (list(torch.split(bins.to(DEV), dims, -1)) if k == "angles" else v.to(DEV) if torch.is_tensor(v) else v)
           for k, v in raw.items()}
    for m in (1, 17, n):
        part = {k: ([a[:m] for a in v] if k == "angles" else v[:m] if torch.is_tensor(v) else (m, head_dim))
                for k, v in dev.items()}
        for d in (part, comp._pack_compressed(part)):
            got = comp.decompress(d).cpu()
            assert got.shape == (m, head_dim)
            torch.testing.assert_close(got, want[:m], atol=0, rtol=0, equal_nan=True)
