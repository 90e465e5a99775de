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


@pytest.mark.parametrize("H,KVH,D,B,q_len,pages,q_dtype,window,part,waves", [
    (14, 2, 64, 4, 1, 512, torch.bfloat16, 4096, 128, 4),   # 65 of 64 tokens: 520 workgroups
    (32, 8, 128, 4, 1, 128, torch.bfloat16, 1024, 128, 4),  # 17 of 64: 544
    (32, 8, 128, 2, 1, 128, torch.bfloat16, 1000, 64, 4),   # 16 of 64, one round
    (28, 4, 128, 4, 1, 298, torch.float32, 1590, 128, 4),   # more than 16 of 64
    (32, 8, 128, 2, 4, 350, torch.bfloat16, 2553, 256, 4),  # 16 rows a tile: of 128
    (32, 8, 128, 32, 4, 512, torch.bfloat16, 128, 192, 4),  # every CU has a row: one partition
    (28, 4, 128, 37, 1, 98, torch.bfloat16, 1043, 384, 4),  # 296 wide ones: a second round
    (28, 4, 128, 16, 1, 224, torch.bfloat16, 2000, 1024, 8),  # 128 wide ones
    (32, 8, 128, 16, 1, 64, torch.bfloat16, 100, 128, 4),   # half the CUs, two tiles a wave: one
    (32, 8, 128, 2, 1, 64, torch.bfloat16, 100, 64, 4),     # fewer rows: two
])
def test_partitions_of_a_window(device, H, KVH, D, B, q_len, pages, q_dtype, window, part, waves):
    """The size of a windowed launch's partitions (256 CUs): one round of workgroups, no more
    partitions than a merge should read, one where that fills the launch."""
    if torch.cuda.get_device_properties(device).multi_processor_count != 256:
        pytest.skip("the sizes are of a 256-CU device")
    cap = 16 * pages
    print(f"[case] H={H}/{KVH} D={D} B={B} q_len={q_len} window={window}", flush=True)
    g = torch.Generator().manual_seed(window)
    lens = [cap, 1, cap - 7][:B] + [int(x) for x in torch.randint(1, cap + 1, (max(0, B - 3),), generator=g)]
    pool = 2 * pages
    q = torch.randn(B, q_len, H, D, generator=g).to(q_dtype)
    kc, vc = (torch.randn(pool, 16, KVH, D, generator=g).to(q_dtype) for _ in range(2))
    table = torch.randint(0, pool, (B, pages), generator=g)
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(B, q_len, H, KVH, D, cap), dtype=torch.uint8,
                     device=device)
    out = paged_attention(q.to(device), kc.to(device), vc.to(device), table.to(device, torch.int32),
                          torch.tensor(lens, dtype=torch.int32, device=device), window=window,
                          workspace=ws)
    hdr = ws[:4 * (64 + 4096)].view(torch.int32).cpu()
    assert (int(hdr[0]), int(hdr[8]), int(hdr[9])) == (2, part, waves), hdr[:16].tolist()
    assert not hdr[64:].any()
    rows = list(range(min(B, 3)))
    ref = dense.paged_attention_f64(q[rows], kc, vc, table[rows], lens[:len(rows)], window=window)
    err = np.abs(out[rows].double().cpu().numpy() - ref).max()
    assert err < (1e-4 if q_dtype == torch.float32 else 2e-2 * np.abs(ref).max())


@pytest.mark.parametrize("H,KVH,D,B,window,q_dtype,kv_dtype,kind", [
    (32, 8, 128, 32, 2544, torch.bfloat16, torch.bfloat16, 2),   # 40,704 tiles
    (32, 8, 128, 32, 2560, torch.bfloat16, torch.bfloat16, 1),   # 40,960
    (28, 4, 128, 32, 3056, torch.float32, torch.float32, 2),     # 24,448
    (28, 4, 128, 32, 3072, torch.float32, torch.float32, 1),
    (32, 8, 128, 32, 3072, torch.float32, torch.bfloat16, 1),    # 49,152
    (28, 4, 128, 64, 3072, torch.float32, torch.bfloat16, 2),
    (14, 2, 64, 192, 4080, torch.bfloat16, torch.bfloat16, 2),   # 97,920
    (14, 2, 64, 192, 4096, torch.bfloat16, torch.bfloat16, 1),
])
def test_window_tiles_that_take_stream_k(device, H, KVH, D, B, window, q_dtype, kv_dtype, kind):
    """The kernel on both sides of the lines in tiles a window shows, over a table past them."""
    pages, cap = 264, 16 * 264
    print(f"[case] H={H}/{KVH} D={D} B={B} window={window} {q_dtype}/{kv_dtype}", flush=True)
    g = torch.Generator(device).manual_seed(window)
    lens = torch.randint(1, cap + 1, (B,), generator=torch.Generator().manual_seed(B)).to(torch.int32)
    lens[0], lens[1], lens[2] = cap, 0, window + 1
    q = torch.randn(B, 1, H, D, generator=g, device=device).to(q_dtype)
    kc, vc = (torch.randn(pages, 16, KVH, D, generator=g, device=device).to(kv_dtype)
              for _ in range(2))
    table = torch.randint(0, pages, (B, pages), generator=torch.Generator().manual_seed(1))
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(B, 1, H, KVH, D, cap), dtype=torch.uint8,
                     device=device)
    out = paged_attention(q, kc, vc, table.to(device, torch.int32), lens.to(device), window=window,
                          workspace=ws)
    assert int(ws[:4].view(torch.int32)) == kind
    ref = dense.paged_attention_f64(q[:3].cpu(), kc.cpu(), vc.cpu(), table[:3], lens[:3].tolist(),
                                    window=window, kv_cast=True)
    err = np.abs(out[:3].double().cpu().numpy() - ref).max()
    assert err < (1e-4 if q_dtype == torch.float32 else 2e-2 * np.abs(ref).max())


@pytest.mark.parametrize("window", [96, 1 << 20, 2 ** 31 - 1])
@pytest.mark.parametrize("H,KVH,D,q_len,q_dtype,kv_dtype,pages", [
    (4, 4, 64, 16, torch.bfloat16, torch.bfloat16, 6),        # the partition kernel
    (28, 4, 128, 1, torch.bfloat16, torch.bfloat16, 6),
    (28, 4, 128, 60, torch.bfloat16, torch.float8_e4m3fn, 6),  # chunks on both prefill kernels
    (6, 2, 96, 60, torch.float32, torch.float32, 4096),
    (6, 2, 96, 2, torch.float32, torch.float32, 6),           # the generic kernel
])
def test_a_window_that_hides_nothing(device, H, KVH, D, q_len, q_dtype, kv_dtype, pages, window):
    """Contexts shorter than the chunk among them: bit for bit the call without a window, up to
    the largest value that a window can take."""
    cap = 16 * pages
    window = max(window, cap)
    print(f"[case] H={H}/{KVH} D={D} q_len={q_len} {q_dtype}/{kv_dtype} window={window}", flush=True)
    g = torch.Generator().manual_seed(q_len)
    lens = torch.tensor([5, 0, 96, 61], dtype=torch.int32, device=device)
    q = torch.randn(4, q_len, H, D, generator=g).to(q_dtype).to(device)
    kc, vc = (torch.randn(32, 16, KVH, D, generator=g).to(kv_dtype).to(device) for _ in range(2))
    table = torch.randint(0, 32, (4, pages), generator=g).to(torch.int32).to(device)
    want = paged_attention(q, kc, vc, table, lens)
    assert torch.equal(paged_attention(q, kc, vc, table, lens, window=window), want)
