"""A graph capture after one eager call on the stream, which a capture cannot
extend by allocating: the eager call leaves a workspace that holds the captured
one, also where the eager call needs none (one split) or less with more tokens,
and at head_dim 64 where it has fewer rows.  Replays between eager work equal
the eager result bit for bit."""
from __future__ import annotations

import pytest
import torch

from turborag_amd.synthetic import permuted_slots

pytestmark = pytest.mark.gpu
B = 16


def _pool(tq, scheme, H, D, N, cuda):
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    prod = scheme == "turbo_prod"
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    g = torch.Generator(device=cuda).manual_seed(710)
    k, v = (torch.randn(N, H, D, generator=g, device=cuda).half() for _ in range(2))
    slots = permuted_slots(N, B, seed=711).to(cuda)
    pool = torch.zeros((N + B - 1) // B * lay.page_size_bytes, dtype=torch.uint8, device=cuda)
    (tq.pack if prod else tq.mse_pack)(k, v, slots, pool, lay, cfg)
    return cfg, lay, slots, pool, g


def _capture(call, warm, later, out, want):
    """call(case, stream) on `warm` eagerly, then `later` captured and replayed."""
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    call(warm, side.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(later, side.cuda_stream)
    for _ in range(3):
        out.fill_(7.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        call(warm, side.cuda_stream)  # eager work on the stream in between
        torch.cuda.synchronize()


@pytest.mark.parametrize("scheme,D,H,warm,later", [
    # (rows, tokens)
    ("turbo_prod", 128, 2, (8, 100), (8, 8192)),
    ("turbo_mse", 128, 2, (8, 76800), (8, 32768)),
    ("turbo_prod", 128, 2, (40, 40000), (40, 20000)),
    ("turbo_prod", 64, 2, (8, 100), (8, 8192)),
    ("turbo_mse", 64, 2, (1, 50), (192, 8192)),
])
def test_slot_mapped(tq, cuda, scheme, D, H, warm, later):
    print(f"[capture {scheme}] D={D} H={H} {warm} then {later}", flush=True)
    tq.release_workspaces()
    cfg, lay, slots, pool, g = _pool(tq, scheme, H, D, max(warm[1], later[1]), cuda)
    q = torch.randn(max(warm[0], later[0]), H, D, generator=g, device=cuda).half()
    outs = {c: torch.zeros(c[0], H, D, dtype=torch.float16, device=cuda) for c in (warm, later)}
    fn = tq.fused_attn_output if scheme == "turbo_prod" else tq.mse_fused_attn_output

    def call(c, stream, out=None):
        fn(q[:c[0]], pool, slots[:c[1]], outs[c] if out is None else out, lay, cfg, *c,
           stream=stream)

    want = torch.zeros_like(outs[later])
    call(later, 0, want)
    _capture(call, warm, later, outs[later], want)
    tq.release_workspaces()


@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
def test_paged_head_dim_64(tq, cuda, scheme):
    """8 rows of one sequence, then 120 row groups."""
    print(f"[capture paged {scheme}]", flush=True)
    tq.release_workspaces()
    H, D, N = 2, 64, 4000
    cfg, lay, slots, pool, g = _pool(tq, scheme, H, D, N, cuda)
    rows = 960
    q = torch.randn(rows, H, D, generator=g, device=cuda).half()
    out = torch.zeros_like(q)
    table = (slots[::B] // B).reshape(1, -1).int().contiguous()
    seq = torch.zeros(rows, dtype=torch.int32, device=cuda)
    lens = torch.randint(1, N + 1, (rows,), generator=g, device=cuda).int()

    def call(n, stream, o=None):
        tq.paged_attn_output(scheme, q[:n], pool, table, seq[:n], lens[:n],
                             (out if o is None else o)[:n], lay, cfg, N, stream=stream)

    want = torch.zeros_like(q)
    call(rows, 0, want)
    _capture(call, 8, rows, out, want)
    tq.release_workspaces()
