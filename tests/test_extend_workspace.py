"""The extend reader's workspace (CPU only: sizes, no launch)."""

import random

import pytest
import torch

from mla_kv_quant_amd import PackedMLAPool, kernels


@pytest.mark.parametrize("D,R", [(512, 64), (256, 32)])
def test_no_batch_asks_for_more_than_the_bound(D, R):
    bound, r = kernels.extend_scratch_bound(D, R), random.Random(D)
    most = 0
    for _ in range(3000):
        B = int(2 ** r.uniform(0, 16))
        rows = kernels.extend_scratch_rows(B, r.choice([1, 16, 40, 128, 4096]), D, R, int(2 ** r.uniform(0, 20)),
                                           B * int(2 ** r.uniform(0, 20)))
        most = max(most, rows)
    assert 0 < most <= bound


@pytest.mark.parametrize("D,R", [(512, 64), (256, 32)])
def test_pool_workspace_follows_the_key_rows_alone(D, R):
    """A captured call keeps reading the buffer that it was captured with: a
    batch of no more key rows, whatever its shape, must not replace it, and finds
    room to split its keys."""
    pool = PackedMLAPool(64, 1, D, R, 2, device="cpu")
    short = pool.extend_workspace(500)
    assert pool.extend_workspace(400) is short and short.shape == (500, D + R)
    ws = pool.extend_workspace(20000)
    for B, H, q, rows in ((1, 16, 96, 19999), (1, 128, 4096, 20000), (64, 16, 1, 6400), (3, 40, 700, 1536), (1, 16, 1, 9)):
        assert pool.extend_workspace(rows) is ws
        assert ws.shape[0] - rows >= kernels.extend_scratch_rows(B, H, D, R, q, rows)
    assert pool.extend_workspace(20001) is not ws


def test_a_plan_needs_longer_keys_where_blocks_nearly_fill_the_card():
    """24 steps of keys (twice the mean) up to 7/8 of the compute units, 64 from
    there. 256 units (the count without a device); 64-key steps, a block per 128
    query rows and sequence."""
    D, R, B, rows = 256, 32, 4, lambda blocks: blocks // 4 * 128
    for blocks, keys, split in ((220, 12 * 64, True), (220, 12 * 64 - 1, False), (224, 32 * 64 - 1, False),
                                (224, 32 * 64, True), (256, 32 * 64 - 1, False), (256, 32 * 64, True)):
        assert (kernels.extend_scratch_rows(B, 1, D, R, rows(blocks), B * keys) > 0) == split, (blocks, keys)


def test_refused_extend_calls_keep_their_errors():
    from mla_kv_quant_amd.extend import packed_mla_extend_fwd

    D, R, H = 512, 64, 16
    pool = PackedMLAPool(64, 1, D, R, 4, device="cpu")
    i32, bf = torch.int32, torch.bfloat16
    a = dict(q=torch.zeros(6, H, D + R, dtype=bf), k=torch.zeros(6, D + R, dtype=bf), o=torch.zeros(6, H, D, dtype=bf),
             pool=pool, layer_id=0, qo_indptr=torch.zeros(4, dtype=i32), kv_indptr=torch.zeros(4, dtype=i32),
             kv_indices=torch.zeros(3, dtype=i32), prefix_lens=torch.zeros(3, dtype=torch.int64),
             req_pool_indices=torch.zeros(3, dtype=torch.int64), max_q_len=6, sm_scale=0.1, prefix_lens_cpu=[400] * 3)
    with pytest.raises(ValueError, match="q must have 3 dims"):
        packed_mla_extend_fwd(**dict(a, q=a["q"].reshape(-1)))
    with pytest.raises(ValueError, match="shorter than the batch"):
        packed_mla_extend_fwd(**dict(a, qo_indptr=a["qo_indptr"][:0]))
