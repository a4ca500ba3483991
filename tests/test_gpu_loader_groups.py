"""load_layers over the layer placements its grouping looks at: pages that
follow one another on both sides (one copy per group), on one side only, in
another order, in two buffers, in pageable memory, and more bytes than one
group takes; every placement equals the one-layer dequant of the same pages."""
from __future__ import annotations

import pytest
import torch

from turborag_amd.synthetic import kv_tokens_major, permuted_slots

pytestmark = pytest.mark.gpu


def _placed(pools, how):
    """The layers' tensors in the memory `how` describes (host or device like pools)."""
    L, n = len(pools), pools[0].numel()
    new = lambda k: (torch.empty(k * n, dtype=torch.uint8, pin_memory=how["pin"])  # noqa: E731
                     if pools[0].is_cpu else torch.empty(k * n, dtype=torch.uint8, device="cuda"))
    if how["place"] == "one":
        rows = list(new(L).view(L, n))
    elif how["place"] == "two":
        rows = list(new(L - 2).view(L - 2, n)) + list(new(2).view(2, n))
    elif how["place"] == "reversed":
        rows = list(new(L).view(L, n))[::-1]
    else:
        rows = [new(1) for _ in range(L)]
    return rows


@pytest.mark.parametrize("scheme,D,L,N,host,dev,pin", [
    ("turbo_prod", 128, 5, 700, "one", "one", True),
    ("turbo_mse", 64, 5, 700, "one", "one", True),
    ("turbo_prod", 64, 5, 700, "two", "one", True),
    ("turbo_mse", 128, 5, 700, "one", "two", True),
    ("turbo_prod", 128, 5, 700, "reversed", "one", True),
    ("turbo_prod", 128, 5, 700, "reversed", "reversed", True),
    ("turbo_mse", 64, 5, 700, "each", "each", True),
    ("turbo_mse", 128, 5, 700, "one", "one", False),
    ("turbo_prod", 128, 7, 20000, "one", "one", True),   # 37 MB: two groups
])
def test_placements(tq, cuda, scheme, D, L, N, host, dev, pin):
    print(f"[loader groups {scheme}] D={D} {L} x {N} host={host} dev={dev} pin={pin}", flush=True)
    H, B = 2, 16
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    prod = scheme == "turbo_prod"
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    slots = permuted_slots(N, B, seed=670).to(cuda)
    pages = int(slots.max()) // B + 1
    k, v = (x.to(cuda) for x in kv_tokens_major(N, H, D, seed=671))
    pools = []
    for layer in range(L):
        p = torch.zeros(pages * lay.page_size_bytes, dtype=torch.uint8, device=cuda)
        (tq.pack if prod else tq.mse_pack)(k.roll(layer, 0).contiguous(), v.roll(layer, 0).contiguous(),
                                           slots, p, lay, cfg)
        pools.append(p)
    hosts = _placed([p.cpu() for p in pools], {"place": host, "pin": pin})
    for h, p in zip(hosts, pools):
        h.copy_(p.cpu())
    devs = _placed(pools, {"place": dev, "pin": False})
    for d in devs:
        d.zero_()
    new = lambda: [torch.full((1, H, N, D), 7.0, dtype=torch.float16, device=cuda)  # noqa: E731
                   for _ in range(L)]
    oks, ovs, wks, wvs = new(), new(), new(), new()
    copy = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(2):  # the second call reuses the device pages
        tq.load_layers(scheme, hosts, devs, slots, oks, ovs, lay, cfg, N,
                       copy_stream=copy.cuda_stream,
                       compute_stream=torch.cuda.current_stream().cuda_stream)
    for p, wk, wv in zip(pools, wks, wvs):
        (tq.dequant_hnd if prod else tq.mse_dequant_hnd)(p, slots, wk, wv, lay, cfg, N)
    torch.cuda.synchronize()
    for layer in range(L):
        assert torch.equal(devs[layer], pools[layer]), layer
        assert torch.equal(oks[layer], wks[layer]) and torch.equal(ovs[layer], wvs[layer]), layer


@pytest.mark.parametrize("shared", ["all", "pairs", "half"])
def test_shared_outputs(tq, cuda, shared):
    """Layers that write one output buffer, or overlapping ones, go in order
    whatever the placement of their pages: the last one's values stay."""
    print(f"[loader groups] outputs shared: {shared}", flush=True)
    H, B, D, L, N = 2, 16, 64, 6, 900
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    lay = tq.make_mse_layout_for(cfg)
    slots = permuted_slots(N, B, seed=672).to(cuda)
    pages = int(slots.max()) // B + 1
    k, v = (x.to(cuda) for x in kv_tokens_major(N, H, D, seed=673))
    pools = torch.zeros(L, pages * lay.page_size_bytes, dtype=torch.uint8, device=cuda)
    for layer in range(L):
        tq.mse_pack(k.roll(layer, 0).contiguous(), v.roll(layer, 0).contiguous(), slots,
                    pools[layer], lay, cfg)
    host = torch.empty(pools.shape, dtype=torch.uint8, pin_memory=True)
    host.copy_(pools)
    n = N * H * D
    flat = torch.full((2 * L * n,), 7.0, dtype=torch.float16, device=cuda)
    want = flat.clone()
    at = [{"all": 0, "pairs": l // 2 * n, "half": l * n // 2}[shared] for l in range(L)]
    out = lambda buf, l, side: buf[side * L * n + at[l]:][:n].view(1, H, N, D)  # noqa: E731
    for layer in range(L):
        tq.mse_dequant_hnd(pools[layer], slots, out(want, layer, 0), out(want, layer, 1), lay, cfg, N)
    copy = torch.cuda.Stream()
    devs = torch.zeros_like(pools)
    torch.cuda.synchronize()
    tq.load_layers("turbo_mse", list(host), list(devs), slots, [out(flat, l, 0) for l in range(L)],
                   [out(flat, l, 1) for l in range(L)], lay, cfg, N, copy_stream=copy.cuda_stream,
                   compute_stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(flat, want)
