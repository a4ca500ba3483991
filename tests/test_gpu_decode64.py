"""The matrix-core decode at head_dim 64: chunk, wave and split edges, partial
row groups, unmapped tokens, and query magnitudes outside the fp16 range,
against the fp64 oracle.

Bound: the kernel's fp32 sums and hi/lo operands are exact to ~2^-20 of a row,
far below fp16's half ulp, so an output differs from the correctly rounded
exact result by at most one fp16 ulp of its row's largest element (both sides
of a rounding boundary)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from turborag_amd.synthetic import as_u16, kv_tokens_major, permuted_slots

pytestmark = pytest.mark.gpu
D, B = 64, 16


def _row_ulps(got16: np.ndarray, ref: np.ndarray) -> float:
    g = got16.reshape(-1, D).astype(np.float64)
    r = ref.reshape(-1, D)
    m = np.abs(r).max(axis=1).astype(np.float16)
    ulp = np.nextafter(m, np.float16(np.inf)).astype(np.float64) - m.astype(np.float64)
    return float((np.abs(g - r.astype(np.float16).astype(np.float64)).max(axis=1) / ulp).max())


def _check(tq, oracle, cuda, scheme, q, k, v, slots, all_slots):
    Q, H, N = q.shape[0], q.shape[1], k.shape[0]
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    prod = scheme == "turbo_prod"
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    pages = int(all_slots.max()) // B + 1
    pack = oracle.prod_pack if prod else oracle.mse_pack
    pool = pack(as_u16(k), as_u16(v), all_slots.numpy(), pages, B)
    f64 = oracle.prod_attention_f64 if prod else oracle.mse_attention_f64
    ref = f64(as_u16(q), pool, slots.numpy(), B)
    out = torch.full((Q, H, D), 7.0, dtype=torch.float16, device=cuda)
    fn = tq.fused_attn_output if prod else tq.mse_fused_attn_output
    fn(q.to(cuda), torch.from_numpy(pool).to(cuda), slots.to(cuda), out, lay, cfg, Q, N)
    torch.cuda.synchronize()
    u = _row_ulps(out.cpu().numpy(), ref)
    print(f"    {u:.2f} row-max ulps", flush=True)
    assert u <= 1.0


@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
@pytest.mark.parametrize("Q,H,N", [(1, 1, 1), (1, 2, 31), (7, 2, 32), (8, 3, 33), (9, 2, 256),
                                   (17, 1, 257), (7, 2, 6001), (8, 8, 2049),
                                   (16, 128, 1500)])  # logits up to ~60: K's lo parts matter
def test_edges(tq, oracle, cuda, scheme, Q, H, N):
    print(f"[decode64 {scheme}] Q={Q} H={H} N={N}", flush=True)
    k, v = kv_tokens_major(N, H, D, seed=N)
    slots = permuted_slots(N, B, seed=N + 1)
    _check(tq, oracle, cuda, scheme, kv_tokens_major(Q, H, D, seed=N + 2)[0], k, v, slots, slots)


@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
def test_unmapped_tokens(tq, oracle, cuda, scheme):
    N, H = 700, 2
    print(f"[decode64 holes {scheme}]", flush=True)
    k, v = kv_tokens_major(N, H, D, seed=5)
    slots = permuted_slots(N, B, seed=6)
    holes = slots.clone()
    holes[::7] = -1
    holes[256:600] = -1  # one whole split and most of the next
    _check(tq, oracle, cuda, scheme, kv_tokens_major(3, H, D, seed=7)[0], k, v, holes, slots)


@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
@pytest.mark.parametrize("q_scale,k_scale", [(2.0 ** 14, 2.0 ** -13), (2.0 ** -11, 2.0 ** 10)])
def test_query_magnitudes(tq, oracle, cuda, scheme, q_scale, k_scale):
    """Rotated queries past fp16's largest value, and queries and keys whose
    product is ordinary but whose own sizes are far from 1: the logits, and so
    the outputs, are those of scale 1.  (|k| < 50 before its scale, outlier
    channels included, so the scaled keys stay finite in fp16.)"""
    N, H, Q = 500, 2, 8
    print(f"[decode64 magnitude {scheme}] {q_scale:g} {k_scale:g}", flush=True)
    k, v = kv_tokens_major(N, H, D, seed=8)
    q = (kv_tokens_major(Q, H, D, seed=9)[0].float().clamp(-3.9, 3.9) * q_scale)
    d = torch.arange(D)
    for h in range(H):  # a row whose rotation is one spike of 8 x its entries
        q[0, h] = (1 - 2 * ((d + h) % 2)).float() * q_scale
    _check(tq, oracle, cuda, scheme, q.half(), (k.float() * k_scale).half(), v,
           permuted_slots(N, B, seed=10), permuted_slots(N, B, seed=10))


@pytest.mark.parametrize("scheme,H,lens,widths", [
    ("turbo_prod", 2, [3000, 700, 256, 1, 1500], [8, 3, 5, 1, 2]),  # units of 4, 3, 2 and 1 positions
    ("turbo_mse", 2, [3000, 700, 256, 1, 1500], [8, 3, 5, 1, 2]),
    ("turbo_prod", 1, [31, 33, 255], [1, 4, 6]),
    ("turbo_mse", 8, [2049, 17], [3, 1]),
])
def test_paged(tq, oracle, cuda, scheme, H, lens, widths):
    """The batched paged decode: every row over its causal token range."""
    from turborag_amd.batched import PagedBatch
    print(f"[decode64 paged {scheme}] H={H} lens={lens} widths={widths}", flush=True)
    b = PagedBatch(tq, scheme, lens, widths, kv_heads=H, q_heads=8 * H, head_dim=D, seed=640,
                   device=cuda)
    b.append_new_tokens(seed=641)
    query, row_seq, row_len = b.decode_rows(seed=642)
    out = torch.full_like(query, 7.0)
    b.attention(query, row_seq, row_len, b.block_tables(), out)
    torch.cuda.synchronize()
    pool, q = b.pool.cpu().numpy(), as_u16(query)
    f64 = oracle.prod_attention_f64 if scheme == "turbo_prod" else oracle.mse_attention_f64
    refs, r = [], 0
    for s, (L, w) in enumerate(zip(lens, widths)):
        for j in range(w):
            refs.append(f64(q[r:r + 8].copy(), pool, b.slots_of(s, L + j + 1), B))
            r += 8
    u = _row_ulps(out.cpu().numpy(), np.concatenate(refs))
    print(f"    {u:.2f} row-max ulps", flush=True)
    b.close()
    assert u <= 1.0


@pytest.mark.parametrize("Q,H,N,scale", [(1, 1, 17, 1.0), (8, 2, 127, 1.0), (9, 3, 128, 1.0),
                                         (17, 2, 1001, 1.0), (8, 2, 300, 2.0 ** 13),
                                         (8, 2, 300, 2.0 ** -11)])
def test_logits(tq, oracle, cuda, Q, H, N, scale):
    """The turbo_prod logits entry on the matrix cores: wave and workgroup
    edges, unaligned rows, unmapped tokens, query magnitudes; within 1e-5 of the
    row's largest logit (fp32 sums of hi/lo parts: ~2^-22 per term)."""
    print(f"[logits64] Q={Q} H={H} N={N} scale={scale:g}", flush=True)
    k, v = kv_tokens_major(N, H, D, seed=20 + N)
    slots = permuted_slots(N, B, seed=21 + N)
    q = (kv_tokens_major(Q, H, D, seed=22 + N)[0].float().clamp(-7.9, 7.9) * scale)
    d = torch.arange(D)
    for h in range(H):  # a row whose rotation is one spike of 8 x its entries
        q[0, h] = (1 - 2 * ((d + h) % 2)).float() * 7.9 * scale
    q = q.half()
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    lay = tq.make_layout_for(cfg)
    pool = oracle.prod_pack(as_u16(k), as_u16(v), slots.numpy(), int(slots.max()) // B + 1, B)
    if N > 100:
        slots[::9] = -1
    _, ref = oracle.prod_attention_f64(as_u16(q), pool, slots.numpy(), B, want_logits=True)
    out = torch.full((Q, H, N), 7.0, device=cuda)
    tq.fused_attn_logits(q.to(cuda), torch.from_numpy(pool).to(cuda), slots.to(cuda), out, lay, cfg,
                         Q, N)
    torch.cuda.synchronize()
    got, ref = out.cpu().double().numpy().reshape(-1, N), ref.reshape(-1, N)
    live = slots.numpy() >= 0
    assert np.all(np.isneginf(got[:, ~live]))
    got, ref = got[:, live], ref[:, live]
    err = (np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)).max()
    print(f"    rel err {err:.2e}", flush=True)
    assert err < 1e-5
