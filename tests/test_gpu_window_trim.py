"""Sink + window caches with invalid rows in the attention's key range: the ring has wrapped and
a trim then took more rows than the next step appends, so rows that were overwritten and trimmed
lie between the valid ones and the attention masks.  (In the steady state of a decode loop every
row is valid and nothing is masked.)  Against the oracle's cache, over the single-buffer, the
two-buffer and the several-sequence kernels."""

import numpy as np
import pytest

from mirror_sd_amd import synth
from mirror_sd_amd.config import DFlashConfig
from oracle import dflash_oracle as O
from parity_util import assert_close_fp16, torch_tensors

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# steps: (new rows, rows trimmed after the block, masked): the block's own rows and more
@pytest.mark.parametrize("n_seq,heads,kv,B,sink,window,steps", [
    (1, 4, 2, 8, 4, 24, ((30, 17, False), (2, 13, True), (1, 8, True), (40, 8, False))),
    # just wrapped: the range is shorter than the ring, its first rows invalid
    (1, 4, 2, 8, 4, 24, ((23, 20, False), (3, 8, True))),
    # trimmed into the sink rows
    (1, 4, 2, 8, 4, 24, ((23, 26, False), (1, 8, True))),
    # chunks of several LDS stages in two buffers, 3 and 5 query tiles
    (1, 24, 8, 32, 64, 6400, ((7000, 732, False), (200, 32, True))),
    (1, 40, 8, 32, 64, 6400, ((7000, 732, False), (200, 32, True))),
    # several sequences: the single buffer, and the ring of key blocks (four query tiles)
    (2, 8, 4, 8, 4, 40, ((60, 30, False), (3, 8, True))),
    (3, 32, 8, 32, 8, 200, ((300, 122, False), (20, 32, True), (150, 32, False))),
])
def test_trimmed_window_matches_oracle(n_seq, heads, kv, B, sink, window, steps):
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = DFlashConfig(hidden_size=256, num_hidden_layers=1, intermediate_size=512,
                       num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                       vocab_size=1024, block_size=B, mask_token_id=1023)
    t = synth.make_weights_numpy(cfg, seed=21)
    W = O.OracleWeights(cfg, t)
    noise = np.stack([O.embed(W, np.array([3 + s] + [1023] * (B - 1), dtype=np.int32))
                      for s in range(n_seq)]).astype(np.float16)
    total = sum(s[0] for s in steps)
    th_all = synth.np_normal(21, f"trim.{heads}.{window}", (n_seq, total, 5 * 256), 1.0, np.float16)
    m = DFlashDraftModel(cfg, max_ctx=total + B, max_block=B, max_seqs=n_seq)
    m.load_weights(torch_tensors(t, "cuda"))
    cache = m.make_cache(sink, window)
    ocache = [[O.OracleKVCache(sink, window)] for _ in range(n_seq)]
    r0, appended = 0, 0
    for i, (C, trim, masked) in enumerate(steps):
        th = th_all[:, r0:r0 + C]
        r0 += C
        appended += C + B
        out = m(torch.from_numpy(noise), torch.from_numpy(th), cache=cache)
        torch.cuda.synchronize()
        for s in range(n_seq):
            ref = O.draft_forward(W, noise[s], th[s], cache=ocache[s], fp16=True)
            assert_close_fp16(out[s].float().cpu().numpy(), ref, what=f"step {i} sequence {s}")
            assert appended > sink + window
            assert (ocache[s][0].keys.shape[1] < sink + window) == masked, (i, s)
            ocache[s][0].trim(trim)
        for c in cache:
            c.trim(trim)
    m.close()
