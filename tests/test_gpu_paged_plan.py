"""Paged steps around the limits of the split workgroups' own plan: up to 256
row groups each workgroup plans the step for itself (with a pass per segment
while the step has no more passes than segments), past them the plan kernel
does.  Every row group equals the slot-mapped decode over its sequence's
tokens (two correct fp16 results: within 2e-3 of a row's largest element)."""
from __future__ import annotations

import pytest
import torch

from turborag_amd.batched import PagedBatch
from turborag_amd.synthetic import uniform_ints

pytestmark = pytest.mark.gpu


def _widths(groups: int, seed: int) -> list[int]:
    w, left = [], groups
    for x in uniform_ints(seed, groups, 1, 9):
        if left <= 0:
            break
        w.append(int(min(x, left)))
        left -= w[-1]
    return w


@pytest.mark.parametrize("scheme,D,H,groups,longest", [
    ("turbo_prod", 128, 2, 256, 120),   # at the limit, a pass per unit
    ("turbo_mse", 128, 2, 257, 120),    # past it: the plan kernel
    ("turbo_prod", 64, 2, 255, 700),
    ("turbo_mse", 64, 1, 259, 700),
    ("turbo_prod", 128, 4, 5, 2600),    # fewer passes than segments: one each
    ("turbo_mse", 128, 8, 13, 2600),    # more passes than the 32 segments of a head
    ("turbo_prod", 128, 1, 1, 32768),   # one unit over 128 segments
    ("turbo_prod", 64, 8, 1, 8192),     # as many passes as segments
    ("turbo_prod", 64, 8, 1, 8193),     # one more
])
def test_plan_limits(tq, cuda, scheme, D, H, groups, longest):
    print(f"[paged plan {scheme}] D={D} H={H} groups={groups} longest={longest}", flush=True)
    widths = _widths(groups, 650 + groups)
    lens = [int(x) for x in uniform_ints(651 + groups, len(widths), 1, longest)]
    lens[-1] = longest - widths[-1]
    b = PagedBatch(tq, scheme, lens, widths, kv_heads=H, q_heads=8 * H, head_dim=D, seed=652,
                   device=cuda)
    b.append_new_tokens(seed=653)
    query, row_seq, row_len = b.decode_rows(seed=654)
    assert query.shape[0] == 8 * groups
    out, ref = torch.full_like(query, 7.0), torch.zeros_like(query)
    b.attention(query, row_seq, row_len, b.block_tables(), out)
    fn = tq.fused_attn_output if scheme == "turbo_prod" else tq.mse_fused_attn_output
    r = 0
    for s, (L, w) in enumerate(zip(lens, widths)):
        slots = torch.from_numpy(b.slots_of(s, L + w)).to(cuda)
        for j in range(w):
            fn(query[r:r + 8].contiguous(), b.pool, slots, ref[r:r + 8], b.layout, b.cfg, 8,
               L + j + 1)
            r += 8
    torch.cuda.synchronize()
    o, e = out.float().reshape(-1, D), ref.float().reshape(-1, D)
    err = ((o - e).abs().amax(1) / e.abs().amax(1)).max().item()
    print(f"    worst rel diff {err:.3e}", flush=True)
    b.close()
    assert err < 2e-3
