"""Queries, keys and values given as views (a model's transposed projections) are read where
they lie: the same bits as from contiguous copies, on every route and type, with strides that
take vector loads and strides that do not, and with views that share memory with what the
call writes."""
import pytest
import torch

from miniserve_amd import PagedAttention, paged_attention

pytestmark = pytest.mark.gpu

F32, F16, BF16, FP8 = torch.float32, torch.float16, torch.bfloat16, torch.float8_e4m3fn


def views(x, pad=5):
    """Views equal to x [B, T, H, D]: transposed, rows padded by `pad`, batch-expanded."""
    B, T, H, D = x.shape
    yield "transposed", x.transpose(1, 2).contiguous().transpose(1, 2)
    wide = x.new_zeros(B, T, H, D + pad)
    wide[..., :D] = x
    yield "padded", wide[..., :D]
    flat = x.new_zeros(B, T, H * D + 8)
    flat[..., 1:1 + H * D] = x.flatten(2)
    yield "base off by an element", flat[..., 1:1 + H * D].unflatten(2, (H, D))
    yield "token-major", x.permute(1, 2, 0, 3).contiguous().permute(2, 0, 1, 3)


@pytest.mark.parametrize("H,KVH,D,q_len,ctx,q_dtype,kv_dtype", [
    (28, 4, 128, 130, 700, BF16, BF16),    # the copying prefill kernel
    (14, 2, 64, 300, 300, F16, FP8),       # its register-staged form
    (16, 4, 128, 300, 4000, F32, F32),     # the any-layout kernel
    (24, 8, 96, 200, 3000, BF16, BF16),    # the same, 16-bit
    (8, 2, 64, 3, 200, BF16, BF16),        # the partition kernel: copied first
])
def test_query_views(device, H, KVH, D, q_len, ctx, q_dtype, kv_dtype):
    g = torch.Generator(device).manual_seed(D + q_len)
    B, pages = 2, -(-ctx // 16)
    q = torch.randn(B, q_len, H, D, generator=g, device=device).to(q_dtype)
    kc, vc = (torch.randn(B * pages, 16, KVH, D, generator=g, device=device).to(kv_dtype)
              for _ in range(2))
    table = torch.randperm(B * pages, device=device).to(torch.int32).view(B, pages)
    lens = torch.tensor([ctx, ctx - 3], dtype=torch.int32, device=device)
    want = paged_attention(q, kc, vc, table, lens)
    for name, v in views(q):
        print(f"[case] query {name} H={H}/{KVH} D={D} {q_dtype}/{kv_dtype}", flush=True)
        assert torch.equal(v, q)
        got = paged_attention(v, kc, vc, table, lens)
        assert torch.equal(got, want)
    one = q[:1].expand(B, -1, -1, -1)  # stride 0
    assert torch.equal(paged_attention(one, kc, vc, table, lens),
                       paged_attention(one.contiguous(), kc, vc, table, lens))
    base = q.transpose(1, 2).contiguous()  # the output over the query's own memory
    out = base.view(B, q_len, H, D)
    assert torch.equal(paged_attention(base.transpose(1, 2), kc, vc, table, lens, out=out), want)


@pytest.mark.parametrize("src,dst", [(F16, F16), (BF16, FP8), (F32, BF16), (F32, F32)])
@pytest.mark.parametrize("D,T", [(128, 37), (64, 1), (6, 5)])
def test_write_kv_views(device, src, dst, D, T):
    KVH, B, pages = 3, 2, 5
    g = torch.Generator(device).manual_seed(D + T)
    k, v = (torch.randn(B, T, KVH, D, generator=g, device=device).to(src) for _ in range(2))
    table = torch.randperm(B * pages, device=device).to(torch.int32).view(B, pages)
    pa = PagedAttention(KVH, KVH, D, num_blocks=B * pages, block_size=16, dtype=src, kv_dtype=dst,
                        device=device)
    bits = {F32: torch.int32, F16: torch.int16, BF16: torch.int16, FP8: torch.int8}[dst]
    want = pa.allocate_kv_cache()
    pa.write_kv(*want, k, v, table, start=[3, 16])
    for (name, kv), (_, vv) in zip(views(k), views(v, pad=8)):
        print(f"[case] write {name} D={D} T={T} {src}->{dst}", flush=True)
        for pair in ((kv, vv), (kv, v), (k, vv)):
            got = pa.allocate_kv_cache()
            pa.write_kv(*got, *pair, table, start=[3, 16])
            for a, b in zip(got, want):
                assert torch.equal(a.view(bits), b.view(bits))


def test_write_kv_from_the_cache_itself(device):
    """Rows moved inside one cache: the source view is copied before anything is written."""
    pa = PagedAttention(2, 2, 64, num_blocks=8, block_size=16, dtype=F16, kv_dtype=F16,
                        device=device)
    kc, vc = (torch.randn(8, 16, 2, 64, device=device).half() for _ in range(2))
    table = torch.arange(8, dtype=torch.int32, device=device)[None]
    k = kc.view(1, 128, 2, 64)[:, 0:60:2]
    v = vc.view(1, 128, 2, 64)[:, 0:60:2]
    want = (k.clone(), v.clone())
    pa.write_kv(kc, vc, k, v, table, start=1)
    assert torch.equal(kc.view(1, 128, 2, 64)[:, 1:31], want[0])
    assert torch.equal(vc.view(1, 128, 2, 64)[:, 1:31], want[1])


@pytest.mark.parametrize("T,name,in_place", [
    (3072, "base off by an element", True), (3073, "base off by an element", False),
    (3073, "transposed", True), (3073, "padded", False)])
def test_large_sources_off_16_bytes_are_copied(device, monkeypatch, T, name, in_place):
    """Rows of 8 x 128 past the line take the vector kernel over a copy unless their strides do."""
    from miniserve_amd import _native as nat

    pa = PagedAttention(8, 8, 128, num_blocks=T // 16 + 1, block_size=16, dtype=F16, kv_dtype=F16,
                        device=device)
    k, v = (torch.randn(1, T, 8, 128, device=device).to(F16) for _ in range(2))
    table = torch.randperm(T // 16 + 1, device=device).to(torch.int32)[None]
    want = pa.allocate_kv_cache()
    pa.write_kv(*want, k, v, table)
    kv = dict(views(k))[name]
    calls = []
    strided = nat.lib().msattn_write_kv_strided
    monkeypatch.setattr(nat.lib(), "msattn_write_kv_strided",
                        lambda *a: calls.append(1) or strided(*a))
    got = pa.allocate_kv_cache()
    pa.write_kv(*got, kv, v, table)
    assert bool(calls) == in_place
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
