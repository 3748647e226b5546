"""GPU parity of the one-token decode over bf16 / f16 K/V (fdecode16_kernel):
float pages of a block pool with rows of unequal length (empty, one token, the
edges of the 16-token step, of the workgroup's 8 steps and of its part), pages
of 16 tokens and of sizes that are no power of two, GQA groups over the 8 a
workgroup holds, the no-allocation entry point, and dense rows whose queries
or strides are unaligned; against 64-bit attention and the generic kernel.  A
call captured without a warm-up (nothing may be allocated) gives the eager
result."""
import pytest
import torch

import vkv
from gpu_util import OPTIONS

pytestmark = pytest.mark.gpu


def reference(q, k, v, scale):
    """q [Hq, D], k / v [Hkv, T, D] -> [Hq, D] in 64 bits (zeros when T = 0)."""
    rep = q.shape[0] // k.shape[0]
    if k.shape[1] == 0:
        return torch.zeros_like(q).double()
    k, v = (x.double().repeat_interleave(rep, 0) for x in (k, v))
    p = torch.softmax((k @ q.double()[:, :, None])[..., 0] * scale, -1)
    return (p[:, None] @ v)[:, 0]


def close(got, ref):
    # 2e-2 for 16-bit outputs and one unit in the last place (bf16: 2^-8)
    assert bool(((got.double() - ref).abs() <= 2e-2 + 2.0 ** -8 * ref.abs()).all())


LENS = [0, 1, 15, 16, 17, 127, 128, 129, 511, 513, 1300]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,D,bs", [(32, 8, 128, 32), (4, 4, 64, 16), (12, 4, 128, 48),
                                         (4, 2, 256, 64), (24, 2, 128, 80), (16, 1, 256, 32)])
def test_float_pages(dtype, Hq, Hkv, D, bs, monkeypatch):
    torch.manual_seed(Hq + D + bs)
    n, scale = len(LENS), D ** -0.5
    nb = (max(LENS) + bs - 1) // bs
    pool = vkv.PagedPool(n * nb, bs, 1, Hkv, D, dtype=vkv.BF16 if dtype == torch.bfloat16 else vkv.F16)
    table = torch.randperm(n * nb, device="cuda").int().view(n, nb).contiguous()
    k, v = (torch.randn((n, nb * bs, Hkv, D), device="cuda").to(dtype) for _ in range(2))
    slots = (table[:, :, None] * bs + torch.arange(bs, device="cuda")).view(-1).int()
    pool.append(0, k.view(-1, Hkv, D), v.view(-1, Hkv, D), slots)
    q = torch.randn((n, Hq, D), device="cuda").to(dtype)
    view = pool.view(0, table, torch.tensor(LENS, dtype=torch.int32, device="cuda"), max(LENS))
    ref = torch.stack([reference(q[i], k[i, :L].transpose(0, 1), v[i, :L].transpose(0, 1), scale)
                       for i, L in enumerate(LENS)])
    for call in range(3):  # the counters are back at zero after every launch
        close(vkv.paged_attention(q, view, scale), ref)
    close(vkv.paged_attention(q, view, scale, noalloc=True), ref)
    for waves in (1, 64, 4096):
        monkeypatch.setattr(OPTIONS, "fdecode_waves", waves)
        close(vkv.paged_attention(q, view, scale), ref)
    monkeypatch.setattr(OPTIONS, "generic_attention", 1)
    close(vkv.paged_attention(q, view, scale), ref)


@pytest.mark.parametrize("T", [16, 130, 2000])
def test_dense_unaligned_queries_and_strided_rows(T):
    """Queries at an odd address, K/V token-major ([B, T, H, D] transposed)."""
    B, Hq, Hkv, D = 2, 8, 2, 128
    torch.manual_seed(T)
    q = torch.randn((B * Hq * D + 1,), device="cuda").bfloat16()[1:].view(B, Hq, 1, D)
    k, v = (torch.randn((B, T, Hkv, D), device="cuda").bfloat16().transpose(1, 2) for _ in range(2))
    out = vkv.scaled_dot_product_attention(q, k, v, D ** -0.5)
    close(out[:, :, 0], torch.stack([reference(q[b, :, 0], k[b], v[b], D ** -0.5) for b in range(B)]))


@pytest.mark.parametrize("masked", [False, True])
def test_capture_without_warm_up(masked):
    """A stream that holds no workspace yet: nothing may be allocated under
    capture, so the decode runs unsplit and a masked chunk generically."""
    B, Hq, Hkv, T, D, L = 1, 8, 2, 3000, 128, 20 if masked else 1
    torch.manual_seed(3)
    q = torch.randn((B, Hq, L, D), device="cuda").bfloat16()
    k, v = (torch.randn((B, Hkv, T, D), device="cuda").bfloat16() for _ in range(2))
    mask = torch.ones((L, T), dtype=torch.bool, device="cuda").tril(T - L) if masked else None
    if masked:  # the generic kernel's own split needs a workspace: none for one part
        k, v, mask = k[:, :, :32], v[:, :, :32], mask[:, :32].contiguous()
    want = vkv.scaled_dot_product_attention(q, k, v, D ** -0.5, mask=mask)
    out = torch.zeros_like(want)
    g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=side):
        vkv.scaled_dot_product_attention(q, k, v, D ** -0.5, mask=mask, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert bool(((out - want).abs() <= 2e-2).all())
