"""Slot-mapped decode with enough row groups that they run as units of up to
four sharing the decoded chunks (units of 4, 3, 2 and 1 groups, partial last
groups, ragged last splits, unmapped tokens), head_dim 128 and 64, against the
fp64 oracle.

Bound: an output differs from the correctly rounded exact result by at most
one fp16 ulp of its row's largest element (the kernel's own arithmetic stays
below half of one)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from turborag_amd.synthetic import as_u16, kv_tokens_major, permuted_slots

pytestmark = pytest.mark.gpu
B = 16


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("scheme,Q,H,N,holes", [
    ("turbo_prod", 16, 128, 1500, False),  # units of two groups
    ("turbo_mse", 13, 128, 1500, False),   # ... the second one partial
    ("turbo_prod", 17, 64, 1500, True),    # three groups
    ("turbo_mse", 32, 64, 1025, True),     # four
    ("turbo_prod", 33, 64, 1500, False),   # four and one
    ("turbo_mse", 41, 64, 2000, False),    # four and two
    ("turbo_prod", 33, 64, 500, True),     # one split: the units write the output
])
def test_units(tq, oracle, cuda, scheme, Q, H, N, holes, D):
    print(f"[decode rows {scheme}] Q={Q} H={H} N={N} D={D}", flush=True)
    oracle.nthreads = 16
    k, v = kv_tokens_major(N, H, D, seed=N)
    slots = permuted_slots(N, B, seed=N + 1)
    pages = int(slots.max()) // B + 1
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    prod = scheme == "turbo_prod"
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    pool = (oracle.prod_pack if prod else oracle.mse_pack)(as_u16(k), as_u16(v), slots.numpy(),
                                                           pages, B)
    if holes:
        slots[::7] = -1
        slots[256:700] = -1
    q = kv_tokens_major(Q, H, D, seed=N + 2)[0]
    f64 = oracle.prod_attention_f64 if prod else oracle.mse_attention_f64
    ref = f64(as_u16(q), pool, slots.numpy(), B).reshape(-1, D)
    out = torch.full((Q, H, D), 7.0, dtype=torch.float16, device=cuda)
    fn = tq.fused_attn_output if prod else tq.mse_fused_attn_output
    fn(q.to(cuda), torch.from_numpy(pool).to(cuda), slots.to(cuda), out, lay, cfg, Q, N)
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(-1, D).astype(np.float64)
    m = np.abs(ref).max(axis=1).astype(np.float16)
    ulp = np.nextafter(m, np.float16(np.inf)).astype(np.float64) - m.astype(np.float64)
    u = (np.abs(got - ref.astype(np.float16).astype(np.float64)).max(axis=1) / ulp).max()
    print(f"    {u:.2f} row-max ulps", flush=True)
    assert u <= 1.0


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("Q,H,N", [(8, 2, 200), (33, 64, 200), (8, 2, 1500)])
def test_output_at_any_half(tq, cuda, Q, H, N, D):
    """An output that starts at an odd half (kernels that write the output
    themselves store 4 and 8 bytes at a time): the bits of an aligned one."""
    print(f"[decode rows, output] Q={Q} H={H} N={N} D={D}", flush=True)
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    lay = tq.make_layout_for(cfg)
    g = torch.Generator(device=cuda).manual_seed(720)
    k, v = (torch.randn(N, H, D, generator=g, device=cuda).half() for _ in range(2))
    q = torch.randn(Q, H, D, generator=g, device=cuda).half()
    slots = torch.arange(N, dtype=torch.int32, device=cuda)
    pool = torch.zeros((N + B - 1) // B * lay.page_size_bytes, dtype=torch.uint8, device=cuda)
    tq.pack(k, v, slots, pool, lay, cfg)
    want = torch.zeros_like(q)
    buf = torch.full((Q * H * D + 2,), 7.0, dtype=torch.float16, device=cuda)
    tq.fused_attn_output(q, pool, slots, want, lay, cfg, Q, N)
    tq.fused_attn_output(q, pool, slots, buf[1:-1].view(Q, H, D), lay, cfg, Q, N)
    torch.cuda.synchronize()
    assert torch.equal(buf[1:-1].view(Q, H, D).view(torch.int16), want.view(torch.int16))
    assert buf[0] == 7.0 and buf[-1] == 7.0
