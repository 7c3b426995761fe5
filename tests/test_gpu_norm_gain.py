"""RMSNorm gains that differ from column to column (a trained model's; the synthetic weights of
the other tests have unit gains) through every kernel that applies a norm as it loads its
input: the stream-K projections and lm_head of one block, the two-m-tile projections of stacked
rows, and the per-step ingest's K|V projection.  Against the CPU oracle, with the tolerance of
the other draft tests (cosine >= 0.9995, max-abs <= 2e-2 in fp16)."""

import numpy as np
import pytest

from mirror_sd_amd import synth
from mirror_sd_amd.config import workload
from oracle import dflash_oracle as O
from parity_util import assert_close_fp16, torch_tensors

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _weights(cfg):
    """Synthetic weights with every norm gain drawn from 1 + 0.3 N(0, 1)."""
    t = synth.make_weights_numpy(cfg, seed=31)
    for name, v in t.items():
        if v.ndim == 1:
            t[name] = (1.0 + 0.3 * synth.np_normal(31, "gain." + name, v.shape)).astype(np.float16)
    return t


@pytest.mark.parametrize("n_seq,block,ctx,vocab", [
    (1, 8, 5, 1024),        # one m-tile, ingest of 5 rows
    (1, 33, 33, 1024),      # two m-tiles with one row in the second, block and ingest
    (2, 20, 40, 1024),      # 40 stacked rows
    (2, 32, 64, 33024),     # two whole m-tiles; a vocabulary that takes the balanced lm_head
    (3, 15, 45, 33024),     # 45 of 64 rows there
    (3, 32, 70, 1024)])     # 96 rows, prompt-sized ingest
def test_column_dependent_norm_gains_match_oracle(n_seq, block, ctx, vocab):
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = workload("tiny").cfg
    cfg.vocab_size = vocab
    t = _weights(cfg)
    W = O.OracleWeights(cfg, t)
    inps = synth.make_batch_inputs_numpy(cfg, block, (ctx,) * n_seq, seed=32)
    m = DFlashDraftModel(cfg, max_ctx=ctx, max_block=block, max_seqs=n_seq)
    m.load_weights(torch_tensors(t, "cuda"))
    for i, inp in enumerate(inps):
        m.ingest_seq(i, torch.from_numpy(inp["target_hidden"]))
    ids = torch.from_numpy(np.stack([inp["ids"] for inp in inps]))
    for _ in range(2):   # the second call meets the counters and keys that the first re-armed
        got, logits, hidden = m.draft_batch(ids=ids, return_logits=True, return_hidden=True)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(got.cpu().numpy(), logits.argmax(-1).cpu().numpy())
    for i, inp in enumerate(inps):
        h_ref, lg_ref, _ = O.draft_block(W, inp["ids"], inp["target_hidden"], fp16=True)
        assert_close_fp16(hidden[i].float().cpu().numpy(), h_ref, what=f"sequence {i} hidden")
        assert_close_fp16(logits[i].cpu().numpy(), lg_ref, what=f"sequence {i} logits")
    m.close()
