"""The one-query scorer splits a unit's query rows over wavefronts in small
launches and not in large ones: both give the same scores and ids, bit for bit
(and the oracle's, which the selection tests compare with small launches)."""

import pytest
import torch

from tests._util import f32_bits
from oracle import nkv_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,r,nb", [(32, 8, 4, 40), (16, 8, 1, 65), (8, 8, 4, 17), (64, 8, 8, 33), (32, 2, 2, 130),
                                         (3, 3, 4, 16), (16, 1, 4, 1)])
def test_small_and_large_launches_score_alike(hq, hkv, r, nb):
    from nanokv_amd.store import SparseKVStore
    parts = min(hq // hkv, 4)
    units = -(-nb // (64 // r)) * hkv
    layers = 2048 // (units * parts) + 2      # past the split's limit
    g = torch.Generator(device="cuda").manual_seed(hq + nb)
    st = SparseKVStore(layers, num_heads=hq, num_kv_heads=hkv, head_dim=128, block_size=64, r=r, cap_blocks=nb + 3,
                       sink_tokens=64, recent_tokens=64)
    st.reps.copy_(torch.randn(st.reps.shape, generator=g, device="cuda"))
    q = torch.randn(layers, 1, hq, 128, generator=g, device="cuda").bfloat16()
    q[0, 0, hq - 1, 5] = float("nan")         # a NaN dot in the last part
    prot = torch.tensor([0], dtype=torch.int32, device="cuda")
    k = min(8, nb)

    def run(layer0, n):
        keys = torch.zeros(n * nb, dtype=torch.int32, device="cuda")
        scores = torch.empty(n, 1, nb, device="cuda")
        ids = torch.full((n, 1, k), -1, dtype=torch.int32, device="cuda")
        vals = torch.empty(n, 1, k, device="cuda")
        st.select(layer0, q[layer0:layer0 + n], nb, prot, 1, k, 0, False, keys, scores, ids, vals)
        assert not keys.any()
        return scores.cpu(), ids.cpu()

    big_scores, big_ids = run(0, layers)
    assert bool(big_scores[0].isnan().all())
    for layer in (0, 1, layers - 1):
        s, i = run(layer, 1)
        assert torch.equal(s.view(torch.int32), big_scores[layer:layer + 1].view(torch.int32))
        assert torch.equal(i, big_ids[layer:layer + 1])
    want = O.block_scores(q[1].float().cpu().numpy(), st.reps[1, :, :nb].float().cpu().numpy(), nb, hkv)
    assert (f32_bits(big_scores[1, 0].numpy()) == f32_bits(want)).all()


@pytest.mark.parametrize("recent", [64, 200, 512, 64 * 70])
def test_protected_rows_are_the_stores_protected_set(recent):
    """The table row of every history length selects as the explicit list does
    (a block named twice in it counts once)."""
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    cfg = M12Config(num_heads=4, num_kv_heads=2, max_model_len=64 * 90, recent_tokens=recent, top_k_blocks=12)
    rt = M12LayerRuntime(0, cfg)
    c = rt._core
    g = torch.Generator(device="cuda").manual_seed(recent)
    rt.store.reps.copy_(torch.randn(rt.store.reps.shape, generator=g, device="cuda"))
    q = torch.randn(1, 4, 128, generator=g, device="cuda").bfloat16()
    rows = rt.store.protected_rows(min(recent // 64, 90)).cpu()
    for nb in (1, 2, 3, 8, 9, 71, 72, 89, 90):
        rt.nblocks_filled = nb
        rt.protected_blocks = {0} | set(range(max(1, nb - recent // 64), nb))
        assert set(rows[nb].tolist()) == rt.protected_blocks
        c._prot_key = None
        got = rt._gpu_select(q)[0]
        dev, n = c.protected_dev()
        assert dev.data_ptr() == rt.store.protected_rows(min(recent // 64, 90))[nb].data_ptr()
        c._prot_dev, listed = torch.tensor(sorted(rt.protected_blocks), dtype=torch.int32, device="cuda"), got
        assert torch.equal(rt._gpu_select(q)[0], listed)
        rt.protected_blocks = rt.protected_blocks | {5}        # a caller's own set: an explicit list
        ids = rt._gpu_select(q)[0]
        assert nb <= 5 or nb - len(rt.protected_blocks) < 1 or 5 not in ids.tolist()
