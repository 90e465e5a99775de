"""Chunked prefill over an fp8 cache on both stagings (tasks of at most 768 keys step by step,
longer ones on the copying schedule): bit for bit the result over the cache widened to the
query type beforehand, which the copying kernel reads as stored."""
import pytest
import torch

from miniserve_amd import kernel_route, paged_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("q_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("pages,lens,window", [
    (48, [768, 33, 129], None), (49, [784, 769, 64], None),   # the rule's line
    (200, [3190, 65, 1], None), (200, [3200, 2000, 700], 700), (200, [3200, 900, 130], 900),
])
def test_fp8_equals_widened(device, D, q_dtype, pages, lens, window):
    H, KVH, q_len, B = 28, 4, 40, len(lens)
    print(f"[case] D={D} {q_dtype} pages={pages} lens={lens} window={window}", flush=True)
    g = torch.Generator(device).manual_seed(pages + D)
    q = torch.randn(B, q_len, H, D, generator=g, device=device).to(q_dtype)
    kc, vc = (torch.randn(B * pages, 16, KVH, D, generator=g, device=device)
              .to(torch.float8_e4m3fn) for _ in range(2))
    table = torch.randperm(B * pages, generator=torch.Generator().manual_seed(1)).view(B, pages)
    table = table.to(device, torch.int32)
    if window is None:
        table[0, 1] = -1  # a hole
    ln = torch.tensor(lens, dtype=torch.int32, device=device)
    assert kernel_route(q, kc, table).startswith("prefill")
    for causal in (True, False):
        got = paged_attention(q, kc, vc, table, ln, causal=causal, window=window)
        want = paged_attention(q, kc.to(q_dtype), vc.to(q_dtype), table, ln, causal=causal,
                               window=window)
        assert torch.equal(got, want)
