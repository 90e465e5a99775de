"""Windowed decodes on the partition kernel: partitions laid from the window's first tile,
against the float64 oracle (the decode tests' bars: 1e-4 in fp32, 2e-2 of the largest output
in 16 bits), for windows that start on and off a tile, shorter and longer than contexts, one
and several query tokens, and every shape of the kernel."""
import numpy as np
import pytest
import torch

from miniserve_amd import _native as nat
from miniserve_amd import paged_attention
from oracle import dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KVH,D,B,q_len,pages,q_dtype,kv_dtype,window", [
    (32, 8, 128, 6, 1, 256, torch.float16, torch.float16, 100),
    (32, 8, 128, 6, 1, 256, torch.float16, torch.float16, 1024),
    (32, 8, 128, 32, 1, 1024, torch.bfloat16, torch.bfloat16, 500),   # a stream-K table
    (28, 4, 128, 6, 1, 400, torch.bfloat16, torch.float8_e4m3fn, 1500),  # the wide shape
    (14, 2, 64, 7, 1, 200, torch.bfloat16, torch.bfloat16, 1),
    (14, 2, 64, 7, 1, 200, torch.bfloat16, torch.bfloat16, 3199),     # all but one key
    (14, 2, 64, 9, 1, 130, torch.float32, torch.float32, 333),
    (28, 4, 128, 5, 4, 300, torch.bfloat16, torch.bfloat16, 257),     # 28 rows: two row tiles
    (4, 4, 128, 5, 9, 300, torch.float32, torch.float32, 64),
])
def test_windowed_decode(device, H, KVH, D, B, q_len, pages, q_dtype, kv_dtype, window):
    cap = 16 * pages
    print(f"[case] H={H}/{KVH} D={D} q_len={q_len} {q_dtype}/{kv_dtype} window={window}", flush=True)
    g = torch.Generator().manual_seed(window + D)
    lens = [int(x) for x in torch.randint(1, cap + 1, (B,), generator=g)]
    lens[:5] = [0, 1, window, min(cap, window + 17), cap]
    counts = [-(-L // 16) for L in lens]
    pool = sum(counts) + 2
    perm = torch.randperm(pool, generator=g).to(torch.int32)
    table = torch.zeros(B, pages, dtype=torch.int32)
    at = 0
    for b, c in enumerate(counts):
        table[b, :c] = perm[at:at + c]
        at += c
    q = torch.randn(B, q_len, H, D, generator=g).to(q_dtype)
    kc, vc = (torch.randn(pool, 16, KVH, D, generator=g).to(kv_dtype) for _ in range(2))
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(B, q_len, H, KVH, D, cap), dtype=torch.uint8,
                     device=device)
    ln = torch.tensor(lens, dtype=torch.int32, device=device)
    ref = dense.paged_attention_f64(q, kc, vc, table.long(), lens, window=window, kv_cast=True)
    for _ in range(3):
        out = paged_attention(q.to(device), kc.to(device), vc.to(device), table.to(device), ln,
                              window=window, workspace=ws)
        hdr = ws[:4 * (64 + 4096)].view(torch.int32).cpu()
        assert int(hdr[0]) == 2 and not hdr[64:].any(), hdr[:16].tolist()
        o = out.double().cpu().numpy()
        assert not o[0].any()
        err = np.abs(o - ref).max()
        assert err < (1e-4 if q_dtype == torch.float32 else 2e-2 * np.abs(ref).max())
