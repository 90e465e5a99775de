"""The any-layout chunked-prefill kernel (csrc/prefill_any.h) against the float64 oracle.

Bars, as the largest error over the largest output: the result's rounding to 16 bits is at
most half a unit in the last place (2^-9 in bf16, 2^-12 in fp16, relative to the value), and
everything before it is held to at least 2^-16, so twice the rounding: 2^-8 and 2^-11 (plus
2^-14 for the weights' split in fp16). In fp32 the sums run over head_dim products and up to
2100 keys, each within 2^-24 of its terms and random in sign: 64 * 2^-24 covers four standard
deviations of sqrt(256) roundings twice.
"""
import numpy as np
import pytest
import torch

from miniserve_amd import _native as nat
from miniserve_amd import kernel_route, paged_attention
from oracle import dense

pytestmark = pytest.mark.gpu

F32, F16, BF16, FP8 = torch.float32, torch.float16, torch.bfloat16, torch.float8_e4m3fn
BAR = {F32: 64 * 2.0 ** -24, F16: 2.0 ** -11 + 2.0 ** -14, BF16: 2.0 ** -8}
ROUTE = "prefill any-layout"


def make(H, KVH, D, lens, q_len, q_dtype, kv_dtype, bs, seed, pad=0):
    g = torch.Generator().manual_seed(seed)
    counts = [max(1, -(-L // bs)) for L in lens]
    pool = sum(counts) + 3
    perm = torch.randperm(pool, generator=g)
    # a table of 2^17 tokens: at that capacity the cost model takes this kernel for the chunks
    # below (an fp32 one with few full row blocks stays on the partition kernel)
    table = torch.zeros(len(lens), (1 << 17) // bs, dtype=torch.int32)
    at = 0
    for b, c in enumerate(counts):
        table[b, :c] = perm[at:at + c]
        at += c
    q = torch.randn(len(lens), q_len, H, D, generator=g).to(q_dtype)
    caches = []
    for _ in range(2):
        c = torch.zeros(pool, bs, KVH, D + pad, dtype=torch.float32)
        c[..., :D] = torch.randn(pool, bs, KVH, D, generator=g)
        caches.append(c.to(kv_dtype))
    return q, caches[0], caches[1], table


def check(device, q, kc, vc, table, lens, D, *, causal=True, window=None, scale=None, shares=None):
    qd, kd, vd, td = (x.to(device) for x in (q, kc, vc, table))
    kd, vd = kd[..., :D], vd[..., :D]
    ln = torch.tensor(lens, dtype=torch.int32, device=device)
    assert kernel_route(qd, kd, td) == ROUTE
    cap = table.shape[1] * kc.shape[1]
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(*q.shape[:2], q.shape[2], kc.shape[2], D, cap),
                     dtype=torch.uint8, device=device)
    outs = [paged_attention(qd, kd, vd, td, ln, causal=causal, window=window, scale=scale,
                            workspace=ws) for _ in range(2)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert not ws[:(64 + 4096) * 4].view(torch.int32)[64:].any(), "tickets not at zero"
    if shares is not None:  # a launch of shares leaves its work list behind the tickets
        tasks = -(-q.shape[1] * q.shape[2] // kc.shape[2] // 128) * kc.shape[2] * q.shape[0]
        work_list = ws[(64 + 4096) * 4:(64 + 4096 + tasks + 2) * 4].view(torch.int32)
        assert bool(work_list.any()) == shares
    ref = dense.paged_attention_f64(q, kc[..., :D], vc[..., :D], table.long(), lens, causal=causal,
                                    window=window, kv_cast=True,
                                    **({} if scale is None else {"scale": scale}))
    o = outs[0].double().cpu().numpy()
    err = float(np.abs(o - ref).max() / max(np.abs(ref).max(), 1e-30))
    print(f"[case] err {err:.2e}", flush=True)
    assert err < BAR[q.dtype]
    return outs[0]


@pytest.mark.parametrize("q_dtype,kv_dtype,D", [
    (q, kv, D) for q, kv in ((F32, F32), (BF16, BF16), (F16, F16), (F16, FP8), (BF16, F32))
    for D in (30, 32, 40, 64, 80, 96, 112, 128, 160, 192, 200, 256)
    if q == F32 or D not in (64, 128)])  # (those are the copying kernel's)
def test_head_sizes(device, q_dtype, kv_dtype, D):
    """Every compiled capacity at its size, below it and off 8-element rows: 381 rows per KV
    head (two blocks and 125 rows) and a context that ends inside a page, one shorter than the
    chunk, and one without keys."""
    lens = [300, 20, 0, 127]
    print(f"[case] D={D} {q_dtype}/{kv_dtype}", flush=True)
    q, kc, vc, table = make(3, 1, D, lens, 127, q_dtype, kv_dtype, 16, D)
    out = check(device, q, kc, vc, table, lens, D)
    assert not out[2].any() and not out[1, :107].any()  # rows that see no key


@pytest.mark.parametrize("q_dtype,kv_dtype", [(F32, BF16), (F32, F16), (F32, FP8), (F16, BF16),
                                              (BF16, F16)])
@pytest.mark.parametrize("H,KVH,D,bs,pad", [(8, 2, 128, 16, 0), (4, 4, 64, 24, 0), (6, 2, 96, 7, 0),
                                            (8, 1, 64, 16, 3)])
def test_layouts(device, q_dtype, kv_dtype, H, KVH, D, bs, pad):
    """Type pairs, pages of 24 and 7 tokens, rows padded off 16-byte boundaries; windows and
    non-causal chunks; a table with holes."""
    q_len, lens = 130, [500, 131]
    print(f"[case] {q_dtype}/{kv_dtype} H={H}/{KVH} D={D} bs={bs} pad={pad}", flush=True)
    q, kc, vc, table = make(H, KVH, D, lens, q_len, q_dtype, kv_dtype, bs, 5, pad)
    check(device, q, kc, vc, table, lens, D)
    check(device, q, kc, vc, table, lens, D, window=70)
    check(device, q, kc, vc, table, lens, D, causal=False, scale=-0.3)
    table[0, 1] = -1
    table[0, 9] = 10 ** 6
    holed = paged_attention(q.to(device), kc.to(device)[..., :D], vc.to(device)[..., :D],
                            table.to(device), torch.tensor(lens, dtype=torch.int32, device=device))
    keep = torch.ones(lens[0], dtype=torch.bool)
    for pg in (1, 9):
        keep[pg * bs:(pg + 1) * bs] = False
    pages = table[0].clamp(0, kc.shape[0] - 1).long()
    flat = [c[..., :D][pages].flatten(0, 1)[:lens[0]].to(q_dtype).double() for c in (kc, vc)]
    k, v = (x.repeat_interleave(H // KVH, 1) for x in flat)
    s = torch.einsum("qhd,khd->hqk", q[0].double(), k) / D ** 0.5
    pos = torch.arange(lens[0])
    seen = (pos[None, :] <= lens[0] - q_len + torch.arange(q_len)[:, None]) & keep[None, :]
    ref = torch.einsum("hqk,khd->qhd", s.masked_fill(~seen, -torch.inf).softmax(-1), v)
    err = (holed[0].double().cpu() - ref).abs().max() / ref.abs().max()
    assert err < BAR[q_dtype]


@pytest.mark.parametrize("H,KVH,D,q_len,lens,q_dtype", [
    (2, 1, 128, 200, [2100], F32),          # four tasks over every CU: shares of a pair
    (8, 8, 64, 380, [1900, 400, 700], F32),  # uneven tasks, three row blocks each
    (6, 2, 96, 256, [2000], BF16),
    (4, 1, 256, 64, [1500, 90], F16),
    (24, 8, 80, 300, [1000, 301], BF16),
])
def test_shares(device, H, KVH, D, q_len, lens, q_dtype):
    """Few tasks over long contexts: the work list split between workgroups and folded."""
    print(f"[case] shares H={H}/{KVH} D={D} q_len={q_len} {q_dtype}", flush=True)
    q, kc, vc, table = make(H, KVH, D, lens, q_len, q_dtype, q_dtype, 16, q_len)
    check(device, q, kc, vc, table, lens, D, shares=True)


@pytest.mark.parametrize("H,KVH,D,q_len,B,cap,q_dtype,kv_dtype", [
    (8, 8, 32, 129, 65, 256, F32, F32),     # 1040 tasks, more than a work list holds
    (8, 8, 32, 129, 65, 256, BF16, BF16),
    (10, 5, 96, 190, 17, 256, F16, F16),    # 255 tasks, not a multiple of 8: about one a CU
    (10, 5, 128, 190, 17, 256, F32, BF16),
    (10, 5, 80, 190, 17, 256, BF16, FP8),
    (21, 3, 200, 60, 20, 128, BF16, BF16),  # 240 tasks of one key-step pair
])
def test_one_task_a_workgroup(device, H, KVH, D, q_len, B, cap, q_dtype, kv_dtype):
    """The launch without shares: tasks dealt to the XCDs, the grid's tail, contexts of every
    kind; the last row block holds part of its 128 rows."""
    print(f"[case] one task H={H}/{KVH} D={D} B={B} {q_dtype}/{kv_dtype}", flush=True)
    lens = [int(x) for x in torch.randint(1, cap + 1, (B,), generator=torch.Generator().manual_seed(D))]
    lens[:4] = [cap, 0, q_len - 1, cap - 1]
    q, kc, vc, table = make(H, KVH, D, lens, q_len, q_dtype, kv_dtype, 16, q_len)
    table = table[:, :cap // 16].contiguous()
    check(device, q, kc, vc, table, lens, D, shares=False)
    check(device, q, kc, vc, table, lens, D, shares=False, window=50)


@pytest.mark.parametrize("q_dtype,rows", [(F32, 120), (BF16, 120)])
def test_keys_past_2_27(device, q_dtype, rows):
    """A context of 2^27 + 4096 tokens whose table repeats one page, its last page apart: keys of
    score 0 and value 1, and a last page whose 4096 keys outweigh them with value 2. Every task
    reads to its end. The softmax in closed form: n keys of weight 1, 4096 of weight e^s."""
    D, bs, n = 8, 4096, 1 << 27
    print(f"[case] {n + bs} keys, {q_dtype}", flush=True)
    kc = torch.zeros(2, bs, 1, D, dtype=q_dtype, device=device)
    vc = torch.ones(2, bs, 1, D, dtype=q_dtype, device=device)
    kc[1], vc[1] = 1.0, 2.0
    table = torch.zeros(1, n // bs + 1, dtype=torch.int32, device=device)
    table[0, -1] = 1
    q = torch.full((1, rows, 1, D), 1.5, dtype=q_dtype, device=device)  # s = 12
    assert kernel_route(q, kc, table) == ROUTE
    lens = torch.tensor([n + bs], dtype=torch.int32, device=device)
    out = paged_attention(q, kc, vc, table, lens, causal=False, scale=1.0)
    w = 4096 * np.exp(12.0)
    want = (n + 2 * w) / (n + w)
    # (every share's sums of ones are whole numbers below 2^24, so exact in fp32)
    assert float((out.double() - want).abs().max()) / want < BAR[q_dtype]


@pytest.mark.parametrize("q_dtype", [F16, BF16])
@pytest.mark.parametrize("D,gap", [(96, 12.0), (32, 16.0), (200, 20.0)])
def test_weights_far_below_the_largest(device, q_dtype, D, gap):
    """An attention sink: key 0 outweighs every other by e^gap and its value is zero, so the
    output is made of weights down to 2^-29 of the largest. (Values of 2^13 keep it a normal
    fp16 number, so that the bar's rounding holds.)"""
    H, KVH, q_len, lens = 3, 1, 127, [300]
    print(f"[case] sink D={D} {q_dtype} gap={gap}", flush=True)
    q, kc, vc, table = make(H, KVH, D, lens, q_len, q_dtype, q_dtype, 16, D)
    at = int(table[0, 0])
    q[..., 0] = 4.0
    kc[..., 0] = 0
    kc[at, 0] = 0
    kc[at, 0, :, 0] = gap / 4.0 * D ** 0.5
    vc *= 2.0 ** 13
    vc[at, 0] = 0
    check(device, q, kc, vc, table, lens, D)
    check(device, q, kc, vc, table, lens, D, causal=False)


@pytest.mark.parametrize("q_dtype", [F32, F16, BF16])
def test_infinite_values_stay_infinite(device, q_dtype):
    """A value of +inf or -inf that every row sees, at dims of their own: infinite there, and the
    finite result elsewhere (weights that the query type holds exactly among them: equal scores)."""
    H, KVH, D, q_len, lens = 3, 1, 96, 127, [300]
    for same in (False, True):
        print(f"[case] infinite values {q_dtype} equal scores {same}", flush=True)
        q, kc, vc, table = make(H, KVH, D, lens, q_len, q_dtype, q_dtype, 16, 7)
        if same:
            kc.zero_()
        qd, kd, td, ld = (x.to(device) for x in (q, kc, table, torch.tensor(lens, dtype=torch.int32)))
        assert kernel_route(qd, kd, td) == ROUTE
        finite = paged_attention(qd, kd, vc.to(device), td, ld, causal=False)
        at = int(table[0, 3])
        vc[at, 5, 0, 10], vc[at, 6, 0, 11] = float("inf"), float("-inf")
        out = paged_attention(qd, kd, vc.to(device), td, ld, causal=False)
        assert bool((out[..., 10] == float("inf")).all()) and bool((out[..., 11] == float("-inf")).all())
        keep = [d for d in range(D) if d not in (10, 11)]
        assert torch.equal(out[..., keep], finite[..., keep])


@pytest.mark.parametrize("H,KVH,D,q_len,q_dtype,cap", [
    (4, 2, 96, 130, BF16, 4096),     # shares and a fold launch
    (28, 4, 128, 130, F32, 4096),
    (10, 5, 80, 190, F16, 256),      # one task a workgroup
])
def test_captured_chunk_replays_with_new_inputs(device, H, KVH, D, q_len, q_dtype, cap):
    """A captured chunk over replays with other lengths, tables and queries in its buffers, eager
    calls on the same workspace between them: each replay the eager call's bits."""
    B = 17 if cap == 256 else 2
    print(f"[case] capture H={H}/{KVH} D={D} {q_dtype} cap={cap}", flush=True)
    g = torch.Generator(device).manual_seed(D)
    gc = torch.Generator().manual_seed(D)
    kc, vc = (torch.randn(512, 16, KVH, D, generator=g, device=device).to(q_dtype) for _ in range(2))
    q = torch.randn(B, q_len, H, D, generator=g, device=device).to(q_dtype)
    table = torch.randint(0, 512, (B, cap // 16), generator=gc).to(device, torch.int32)
    lens = torch.randint(1, cap + 1, (B,), generator=gc).to(device, torch.int32)
    assert kernel_route(q, kc, table) == ROUTE
    ws = torch.zeros(nat.lib().msattn_workspace_bytes(B, q_len, H, KVH, D, cap), dtype=torch.uint8,
                     device=device)
    out = torch.empty_like(q)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        paged_attention(q, kc, vc, table, lens, workspace=ws, out=out)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        paged_attention(q, kc, vc, table, lens, workspace=ws, out=out)
    for _ in range(4):
        q.copy_(torch.randn(q.shape, generator=g, device=device).to(q_dtype))
        table.copy_(torch.randint(0, 512, table.shape, generator=gc).to(torch.int32))
        lens.copy_(torch.randint(0, cap + 1, (B,), generator=gc).to(torch.int32))
        want = paged_attention(q, kc, vc, table, lens, workspace=ws)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
