"""The several-sequence attention with four query tiles (the ring of key blocks) and both merge
kernels against one draft per sequence (the single-sequence kernels): chunks of one to eight key
blocks, partial last blocks and query tiles, a sequence shorter than one block.  Both paths
round at the same points, so the hidden states differ by the order of fp32 sums and the fp16
roundings that it moves through two layers: 2^-9 of the 2-norm."""

import pytest

from mirror_sd_amd import synth
from mirror_sd_amd.config import DFlashConfig
from parity_util import torch_tensors

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def models():
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = DFlashConfig(hidden_size=256, num_hidden_layers=2, intermediate_size=512,
                       num_attention_heads=32, num_key_value_heads=8, head_dim=128,
                       vocab_size=512, block_size=32, target_layer_ids=[1], num_target_layers=4)
    t = torch_tensors(synth.make_weights_numpy(cfg, seed=9), "cuda")
    many = DFlashDraftModel(cfg, max_ctx=9100, max_block=32, max_seqs=8)
    one = DFlashDraftModel(cfg, max_ctx=9100, max_block=32)
    for m in (many, one):
        m.load_weights(t)
    yield many, one
    many.close()
    one.close()


@pytest.mark.parametrize("ctx,B", [((3, 40), 32), ((1, 31, 97, 500, 2000, 64, 7, 333), 32),
                                   ((9000, 4001, 33), 32), ((5000, 4900, 129, 800), 25),
                                   ((6001, 3000), 31),
                                   # 4096 rows (the wide merge) of up to 57 chunks
                                   ((9000, 40, 33, 7), 32)])
def test_ring_matches_single(models, ctx, B):
    many, one = models
    g = torch.Generator().manual_seed(sum(ctx))
    rows = [torch.randn((c, 256), generator=g).to(torch.float16).cuda() for c in ctx]
    ids = torch.randint(0, 512, (len(ctx), B), generator=g, dtype=torch.int32).cuda()
    for s, r in enumerate(rows):
        many.ingest_seq(s, r, fused_context=True)
    _, hidden = many.draft_batch(ids=ids, return_hidden=True)
    for s, r in enumerate(rows):
        _, want = one.draft(ids[s], r, return_hidden=True, fused_context=True)
        got, want = hidden[s].float(), want.float()
        err = float((got - want).norm() / want.norm())
        assert err <= 2.0 ** -9, (ctx, B, s, err)
