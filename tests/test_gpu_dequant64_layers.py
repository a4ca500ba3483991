"""Multi-layer dequant at head_dim 64 (a row per lane, one launch per 64
layers): edges of a wave's 64 rows, more layers than a launch takes, unmapped
tokens, division paths and buffers that fall back to the per-layer kernels,
bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from turborag_amd.synthetic import as_u16, kv_tokens_major, permuted_slots

pytestmark = pytest.mark.gpu
D = 64


@pytest.mark.parametrize("scheme,NL,N,H,B,head_major,holes,shift", [
    ("turbo_prod", 2, 32, 2, 16, False, False, 0),   # one wave's rows exactly
    ("turbo_mse", 3, 33, 2, 16, True, False, 0),     # and two more
    ("turbo_prod", 5, 777, 3, 8, True, True, 0),     # 3 heads: division paths
    ("turbo_mse", 66, 65, 1, 16, False, True, 0),    # two launches
    ("turbo_mse", 2, 300, 2, 7, False, True, 0),     # 7-token blocks
    ("turbo_prod", 2, 300, 1, 7, False, False, 0),   # 490-byte pages: the per-layer kernels
    ("turbo_prod", 2, 300, 2, 16, False, False, 4),  # pools not 16-byte aligned: likewise
])
def test_layers(tq, oracle, cuda, scheme, NL, N, H, B, head_major, holes, shift):
    print(f"[dequant64 layers {scheme}] {NL} x {N} H={H} B={B} head_major={head_major}", flush=True)
    prod = scheme == "turbo_prod"
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim, cfg.block_size = H, D, B
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    slots = permuted_slots(N, B, seed=660 + N)
    pages = int(slots.max()) // B + 1
    pack = oracle.prod_pack if prod else oracle.mse_pack
    pools_np = []
    for layer in range(NL):
        k, v = kv_tokens_major(N, H, D, seed=661 + layer)
        pools_np.append(pack(as_u16(k), as_u16(v), slots.numpy(), pages, B))
    if holes:
        slots[::5] = -1
    pools = []
    for p in pools_np:
        buf = torch.zeros(p.size + shift, dtype=torch.uint8, device=cuda)
        buf[shift:] = torch.from_numpy(p).to(cuda)
        pools.append(buf[shift:])
    shape = (1, H, N, D) if head_major else (N, H, D)
    oks = [torch.full(shape, 7.0, dtype=torch.float16, device=cuda) for _ in range(NL)]
    ovs = [torch.full(shape, 7.0, dtype=torch.float16, device=cuda) for _ in range(NL)]
    tq.dequant_layers(scheme, pools, slots.to(cuda), oks, ovs, lay, cfg, N, head_major=head_major)
    torch.cuda.synchronize()
    fn = oracle.prod_dequant if prod else oracle.mse_dequant
    sl = slots.numpy()
    live, seven = sl >= 0, np.float16(7.0).view(np.uint16)
    for layer in range(NL):
        wk, wv = fn(pools_np[layer], sl, H, D, B)
        for got, want in ((as_u16(oks[layer]), wk), (as_u16(ovs[layer]), wv)):
            if head_major:
                got = got[0].transpose(1, 0, 2)
            assert np.array_equal(got[live], want[live]), layer
            assert np.all(got[~live] == seven), layer


@pytest.mark.parametrize("scheme,head_major", [("turbo_prod", False), ("turbo_mse", True)])
@pytest.mark.parametrize("N", [24575, 24576])
def test_one_large_layer(tq, oracle, cuda, scheme, head_major, N):
    """Both sides of the row count (49,152) from which one layer takes a row per
    lane, with unmapped tokens."""
    H, B = 2, 16
    print(f"[dequant64 one layer {scheme}] N={N} head_major={head_major}", flush=True)
    oracle.nthreads = 16
    prod = scheme == "turbo_prod"
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    slots = permuted_slots(N, B, seed=680)
    k, v = kv_tokens_major(N, H, D, seed=681)
    pool = (oracle.prod_pack if prod else oracle.mse_pack)(as_u16(k), as_u16(v), slots.numpy(),
                                                           int(slots.max()) // B + 1, B)
    slots[::11] = -1
    shape = (1, H, N, D) if head_major else (N, H, D)
    ok = torch.full(shape, 7.0, dtype=torch.float16, device=cuda)
    ov = torch.full_like(ok, 7.0)
    fn = {(True, False): tq.dequant, (False, True): tq.mse_dequant_hnd}[(prod, head_major)]
    fn(torch.from_numpy(pool).to(cuda), slots.to(cuda), ok, ov, lay, cfg,
       *((N,) if head_major else ()))
    torch.cuda.synchronize()
    wk, wv = (oracle.prod_dequant if prod else oracle.mse_dequant)(pool, slots.numpy(), H, D, B)
    live, seven = slots.numpy() >= 0, np.float16(7.0).view(np.uint16)
    for got, want in ((as_u16(ok), wk), (as_u16(ov), wv)):
        if head_major:
            got = got[0].transpose(1, 0, 2)
        assert np.array_equal(got[live], want[live]) and np.all(got[~live] == seven)


@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
@pytest.mark.parametrize("shared", ["both", "keys", "shifted"])
def test_overlapping_outputs(tq, oracle, cuda, scheme, shared):
    """Layers that write one output buffer (or buffers that overlap by some
    rows) are taken in order: the last layer's values."""
    NL, N, H, B = 12, 3001, 2, 16
    print(f"[dequant64 overlap {scheme}] {shared}", flush=True)
    prod = scheme == "turbo_prod"
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim, cfg.block_size = H, D, B
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    slots = permuted_slots(N, B, seed=690)
    pages = int(slots.max()) // B + 1
    pack = oracle.prod_pack if prod else oracle.mse_pack
    pools_np = []
    for layer in range(NL):
        k, v = kv_tokens_major(N, H, D, seed=691 + layer)
        pools_np.append(pack(as_u16(k), as_u16(v), slots.numpy(), pages, B))
    pools = [torch.from_numpy(p).to(cuda) for p in pools_np]
    step = {"both": 0, "keys": 0, "shifted": 100}[shared]  # tokens between two layers' outputs
    kb = torch.full((N + step * (NL - 1), H, D), 7.0, dtype=torch.float16, device=cuda)
    vb = torch.full_like(kb, 7.0)
    oks = [kb[step * layer:step * layer + N] for layer in range(NL)]
    ovs = [vb[step * layer:step * layer + N] if shared != "keys" else torch.full_like(oks[0], 7.0)
           for layer in range(NL)]
    tq.dequant_layers(scheme, pools, slots.to(cuda), oks, ovs, lay, cfg, N)
    torch.cuda.synchronize()
    fn = oracle.prod_dequant if prod else oracle.mse_dequant
    want_k = np.full(kb.shape, np.float16(7.0).view(np.uint16))
    want_v = want_k.copy()
    for layer in range(NL):
        wk, wv = fn(pools_np[layer], slots.numpy(), H, D, B)
        want_k[step * layer:step * layer + N] = wk
        want_v[step * layer:step * layer + N] = wv
        if shared == "keys":
            assert np.array_equal(as_u16(ovs[layer]), wv)
    assert np.array_equal(as_u16(kb), want_k)
    if shared != "keys":
        assert np.array_equal(as_u16(vb), want_v)
