"""Non-finite values past a paged row's length: an infinity in the value row of
a sequence's last new token (its V scale is infinite) reaches the rows that
attend the token and no others.  The rows of the earlier new tokens, rows of a
shorter length in the same group and rows of length 0 have the bits they have
with a finite value there (units of one to four positions, one chunk and many)."""
from __future__ import annotations

import pytest
import torch

from turborag_amd.batched import PagedBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["turbo_prod", "turbo_mse"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_value_past_a_row(tq, cuda, scheme, D, bad):
    lens, widths = [1, 40, 700, 255, 2900, 30], [2, 1, 3, 4, 6, 8]
    print(f"[paged non-finite {scheme}] D={D} {bad}", flush=True)
    b = PagedBatch(tq, scheme, lens, widths, head_dim=D, seed=690, device=cuda)
    new = b.append_new_tokens(seed=691)
    query, row_seq, row_len = b.decode_rows(seed=692)
    whole = torch.tensor([L + w for L, w in zip(lens, widths)], dtype=torch.int32, device=cuda)
    row_len[3] = 0
    row_len[8 * 2 + 5] = 17        # the one row group of sequence 1
    row_len[8 * 6 + 7] = 0         # padding in a group of sequence 3
    tables = b.block_tables()
    want, got = torch.full_like(query, 7.0), torch.full_like(query, 7.0)
    b.attention(query, row_seq, row_len, tables, want)
    pack = tq.pack if scheme == "turbo_prod" else tq.mse_pack
    for s in range(len(lens)):  # the last new token again, with a non-finite value row
        k, v = new[s][0][-1:].clone(), new[s][1][-1:].clone()
        v[..., 5] = bad
        slot = torch.from_numpy(b.slots_of(s, lens[s] + widths[s])[-1:]).to(cuda)
        pack(k.to(cuda), v.to(cuda), slot, b.pool, b.layout, b.cfg)
    b.attention(query, row_seq, row_len, tables, got)
    torch.cuda.synchronize()
    b.close()
    attends = row_len == whole[row_seq.long()]
    assert attends.any() and not attends.all()
    assert torch.equal(got[~attends].view(torch.int16), want[~attends].view(torch.int16))
    assert torch.isfinite(want).all() and (got[row_len == 0] == 0).all()
    if bad == bad:
        assert not torch.isfinite(got[attends]).any()
