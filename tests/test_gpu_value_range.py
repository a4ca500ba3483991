"""Decode over value rows far from magnitude 1: small ones (their weighted
scales lie among fp16's subnormals), magnitudes that grow or fall along the
context, a leading token above a long tail of low weights; the one-group and
unit kernels over a slot map and the paged step, against the fp64 oracle.

Bound: fp16 rounding of the output (half an ulp of its row's largest element,
or of the subnormals) and the kernel's own arithmetic.  At head_dim 64 that is
~2^-20 of a row: 0.55 ulp.  At head_dim 128 the fp16 value levels are off by up
to 9.3e-5: 0.2 ulp more."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from turborag_amd.synthetic import as_u16, permuted_slots

pytestmark = pytest.mark.gpu
B = 16


def _values(kind: str, n: int) -> torch.Tensor:
    """log2 of the tokens' magnitudes."""
    t = torch.arange(n) / n
    return {"small": torch.full((n,), -10.0), "smaller": torch.full((n,), -13.0),
            "smallest": torch.full((n,), -16.0), "growing": -16.0 + 22.0 * t,
            "falling": 6.0 - 22.0 * t}[kind]


@pytest.mark.parametrize("kind", ["small", "smaller", "smallest", "growing", "falling"])
@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
@pytest.mark.parametrize("D,path,Q,H,N", [
    (64, "slots", 8, 2, 2500),    # one row group per workgroup
    (64, "slots", 33, 64, 700),   # units of four and one
    (64, "paged", 8, 2, 2500),
    (64, "paged", 32, 2, 2500),
    (128, "slots", 33, 64, 700),
])
def test_magnitudes(tq, oracle, cuda, scheme, D, path, Q, H, N, kind):
    print(f"[value range {scheme}] D={D} {path} Q={Q} H={H} N={N} {kind}", flush=True)
    oracle.nthreads = 16
    g = torch.Generator().manual_seed(700)
    lead = torch.randn(H, D, generator=g)
    lead /= lead.norm(dim=-1, keepdim=True)
    k = torch.randn(N, H, D, generator=g) * 0.2
    k[N // 3] += 8 * lead  # ~11 nats above the others
    q = (lead * (11 * D ** 0.5 / 8) + 0.1 * torch.randn(Q, H, D, generator=g)).half()
    v = (torch.randn(N, H, D, generator=g) + 1.0) * torch.exp2(_values(kind, N))[:, None, None]
    slots = permuted_slots(N, B, seed=701)
    prod = scheme == "turbo_prod"
    pool = (oracle.prod_pack if prod else oracle.mse_pack)(
        as_u16(k.half()), as_u16(v.half()), slots.numpy(), int(slots.max()) // B + 1, B)
    ref = (oracle.prod_attention_f64 if prod else oracle.mse_attention_f64)(
        as_u16(q), pool, slots.numpy(), B).reshape(-1, D)
    cfg = tq.default_config()
    cfg.num_kv_heads, cfg.head_dim = H, D
    lay = tq.make_layout_for(cfg) if prod else tq.make_mse_layout_for(cfg)
    out = torch.full((Q, H, D), 7.0, dtype=torch.float16, device=cuda)
    qd, pd = q.to(cuda), torch.from_numpy(pool).to(cuda)
    if path == "slots":
        fn = tq.fused_attn_output if prod else tq.mse_fused_attn_output
        fn(qd, pd, slots.to(cuda), out, lay, cfg, Q, N)
    else:
        table = (slots[::B] // B).reshape(1, -1).int().contiguous().to(cuda)
        tq.paged_attn_output(scheme, qd, pd, table,
                             torch.zeros(Q, dtype=torch.int32, device=cuda),
                             torch.full((Q,), N, dtype=torch.int32, device=cuda), out, lay, cfg, N)
    torch.cuda.synchronize()
    m = np.abs(ref).max(axis=1).astype(np.float16)
    ulp = np.nextafter(m, np.float16(np.inf)).astype(np.float64) - m.astype(np.float64)
    got = out.cpu().numpy().reshape(-1, D).astype(np.float64)
    u = (np.abs(got - ref).max(axis=1) / ulp).max()
    print(f"    {u:.3f} row-max ulps", flush=True)
    assert u <= (0.55 if D == 64 else 0.75)
