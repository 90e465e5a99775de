"""Decodes whose block table ends inside the last 1024-token partition take the partition
kernel's wide shape too (eight waves over 1024-token partitions): the workspace header names
it, and the output meets the float64 oracle's bar of the 16-bit decode tests (2e-2 of the
largest output), with contexts that end before, at and inside the short partition."""
import numpy as np
import pytest
import torch

from miniserve_amd import _native as nat
from miniserve_amd import paged_attention
from oracle import dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pages,kv_dtype", [(193, torch.bfloat16), (219, torch.bfloat16),
                                            (255, torch.bfloat16), (219, torch.float8_e4m3fn)])
def test_table_ends_inside_a_partition(device, pages, kv_dtype):
    H, KVH, D, B, cap = 28, 4, 128, 16, 16 * pages
    print(f"[case] {pages} pages {kv_dtype}", flush=True)
    g = torch.Generator().manual_seed(pages)
    lens = [int(x) for x in torch.randint(1, cap + 1, (B,), generator=g)]
    lens[:6] = [0, 1, 3072, 3073, cap, cap - 1]
    counts = [-(-L // 16) for L in lens]
    pool = sum(counts) + 2
    perm = torch.randperm(pool, generator=g).to(torch.int32)
    table = torch.zeros(B, pages, dtype=torch.int32)
    at = 0
    for b, c in enumerate(counts):
        table[b, :c] = perm[at:at + c]
        at += c
    q = torch.randn(B, 1, H, D, generator=g).to(torch.bfloat16)
    kc, vc = (torch.randn(pool, 16, KVH, D, generator=g).to(kv_dtype) for _ in range(2))
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(B, 1, H, KVH, D, cap), dtype=torch.uint8,
                     device=device)
    ln = torch.tensor(lens, dtype=torch.int32, device=device)
    for _ in range(2):
        out = paged_attention(q.to(device), kc.to(device), vc.to(device), table.to(device), ln,
                              workspace=ws)
        hdr = ws[:4 * (64 + 4096)].view(torch.int32).cpu()
        assert (int(hdr[0]), int(hdr[8]), int(hdr[9])) == (2, 1024, 8), hdr[:16].tolist()
        assert not hdr[64:].any()
    ref = dense.paged_attention_f64(q, kc, vc, table.long(), lens, kv_cast=True)
    o = out.double().cpu().numpy()
    assert not o[0].any()
    assert np.abs(o - ref).max() / np.abs(ref).max() < 2e-2
