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


@pytest.mark.parametrize("H,KVH,D,B,pages,kv_dtype,waves", [
    (32, 8, 128, 32, 8, torch.bfloat16, 4),      # one partition: at least half of it
    (32, 8, 128, 32, 31, torch.bfloat16, 4),
    (32, 8, 128, 32, 32, torch.bfloat16, 8),
    (32, 8, 128, 25, 40, torch.bfloat16, 4),     # 200 of 256 CUs
    (32, 8, 128, 26, 40, torch.bfloat16, 8),     # 208
    (28, 4, 128, 65, 40, torch.bfloat16, 4),     # 260: a second round
    (28, 4, 128, 65, 64, torch.bfloat16, 8),     # the same over whole partitions
    (32, 8, 128, 40, 40, torch.float8_e4m3fn, 4),   # fp8 at 4 rows per tile: uncapped
    (32, 8, 128, 48, 35, torch.float8_e4m3fn, 4),
    (32, 8, 128, 48, 36, torch.float8_e4m3fn, 8),
    (28, 4, 128, 32, 111, torch.bfloat16, 4),    # two partitions: 7/8 of both
    (28, 4, 128, 32, 112, torch.bfloat16, 8),
    (14, 2, 64, 40, 128, torch.bfloat16, 4),     # three: the last may hold one page
    (14, 2, 64, 40, 129, torch.bfloat16, 8),
])
def test_tables_that_fill_enough_of_the_shape(device, H, KVH, D, B, pages, kv_dtype, waves):
    """The rule's lines: which tables and launches take the wide shape (256 CUs)."""
    if torch.cuda.get_device_properties(device).multi_processor_count != 256:
        pytest.skip("the lines are of a 256-CU device")
    cap = 16 * pages
    print(f"[case] H={H}/{KVH} D={D} B={B} {pages} pages {kv_dtype}", flush=True)
    g = torch.Generator(device).manual_seed(pages)
    lens = torch.randint(1, cap + 1, (B,), generator=torch.Generator().manual_seed(B)).to(torch.int32)
    lens[0], lens[1] = cap, 0
    q = torch.randn(B, 1, H, D, generator=g, device=device).to(torch.bfloat16)
    kc, vc = (torch.randn(4 * pages, 16, KVH, D, generator=g, device=device).to(kv_dtype)
              for _ in range(2))
    table = torch.randint(0, 4 * pages, (B, pages), generator=torch.Generator().manual_seed(1))
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(B, 1, H, KVH, D, cap), dtype=torch.uint8,
                     device=device)
    out = paged_attention(q, kc, vc, table.to(device, torch.int32), lens.to(device), workspace=ws)
    hdr = ws[:4 * (64 + 4096)].view(torch.int32).cpu()
    assert (int(hdr[0]), int(hdr[9])) == (2, waves) and not hdr[64:].any(), hdr[:16].tolist()
    rows = [0, 1, B - 1]
    ref = dense.paged_attention_f64(q[rows].cpu(), kc.cpu(), vc.cpu(), table[rows],
                                    lens[rows].tolist(), kv_cast=True)
    o = out[rows].double().cpu().numpy()
    assert np.abs(o - ref).max() / np.abs(ref).max() < 2e-2
