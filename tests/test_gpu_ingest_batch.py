"""dfl_ingest_batch against one dfl_ingest_context per sequence: group sizes on both sides of
one and two m-tiles, of a launch's entries and of the per-step limit, in plain and in sink +
window caches.  The cached rows are the same up to the fp16 rounding of sums taken in another
order (a row's m-tile count may change the kernel), row counts and offsets exactly."""

import ctypes

import pytest

from mirror_sd_amd import _lib, synth
from mirror_sd_amd.config import DFlashConfig
from parity_util import torch_tensors

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CFG = dict(hidden_size=256, num_hidden_layers=3, intermediate_size=512, num_attention_heads=4,
           num_key_value_heads=2, head_dim=128, vocab_size=512, block_size=8,
           target_layer_ids=[1, 3], num_target_layers=6)
MAX_SEQS = 9


@pytest.fixture(scope="module")
def models():
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = DFlashConfig(**CFG)
    t = torch_tensors(synth.make_weights_numpy(cfg, seed=5), "cuda")
    pair = [DFlashDraftModel(cfg, max_ctx=256, max_block=8, max_seqs=MAX_SEQS) for _ in range(2)]
    for m in pair:
        m.load_weights(t)
    yield pair
    for m in pair:
        m.close()


@pytest.mark.parametrize("window", [0, 16])
@pytest.mark.parametrize("n_seq,C", [(2, 1), (9, 1), (8, 8), (9, 7), (3, 16), (2, 32), (3, 31),
                                     (2, 33), (2, 70)])
def test_batch_matches_sequences(models, n_seq, C, window):
    a, b = models
    g = torch.Generator().manual_seed(100 * n_seq + C)
    H = CFG["hidden_size"]
    for m in models:
        m.make_cache(4 if window else 0, window)
        for s in range(MAX_SEQS):
            m.select_seq(s)
            _lib.check(m._L.dfl_cache_reset(m._ctx), "dfl_cache_reset")
        m.select_seq(0)
    for step in range(2):
        th = torch.randn((n_seq, C, 2 * H), generator=g).to(torch.float16).cuda()
        assert a._ingest_seqs(th) == C
        for s in range(n_seq):
            b.ingest_seq(s, th[s], reset=False)
    for s in range(n_seq):
        st = []
        for m in models:
            m.select_seq(s)
            n, off = ctypes.c_int32(), ctypes.c_int64()
            _lib.check(m._L.dfl_cache_state(m._ctx, ctypes.byref(n), ctypes.byref(off)), "state")
            m.select_seq(0)
            st.append((n.value, off.value))
        assert st[0] == st[1] == (min(2 * C, 4 + window) if window else 2 * C, 2 * C)
        rows = st[0][0]
        for (ka, va), (kb, vb) in zip(a.cache_tensors(s), b.cache_tensors(s)):
            for x, y in ((ka[:, :rows], kb[:, :rows]), (va[:, :, :rows], vb[:, :, :rows])):
                x, y = x.float(), y.float()
                # one rounding of the Linear's fp16 (2^-11 of the value) through norm and rotation
                assert float((x - y).abs().max()) <= 4 * 2.0 ** -11 * float(y.abs().max())
                assert float((x - y).norm()) <= 2.0 ** -11 * float(y.norm())


def test_batch_rejects(models):
    m = models[0]
    L, ctx, p = m._L, m._ctx, torch.zeros(8, device="cuda").data_ptr()
    for args in ((0, p, 1), (MAX_SEQS + 1, p, 1), (2, None, 1), (2, p, -1), (2, p, 100000)):
        m.make_cache(0, 0)
        assert L.dfl_ingest_batch(ctx, *args, None) in (_lib.DFL_EINVAL, _lib.DFL_ERANGE)


@pytest.mark.parametrize("n_seq,C", [(3, 70), (2, 33), (3, 20)])
def test_batch_of_strided_rows(models, n_seq, C):
    """The newest rows of a longer buffer: the cached rows of a contiguous copy, bit for bit; a
    step too long to share its launches reads them in place, without a copy of the batch."""
    a, b = models
    g = torch.Generator().manual_seed(C)
    buf = torch.randn((n_seq, 200, 2 * CFG["hidden_size"]), generator=g).to(torch.float16).cuda()
    th = buf[:, -C:]
    for m in models:
        m.make_cache(0, 0)
        for s in range(MAX_SEQS):
            m.select_seq(s)
            _lib.check(m._L.dfl_cache_reset(m._ctx), "dfl_cache_reset")
        m.select_seq(0)
    b._ingest_seqs(th.contiguous())
    torch.cuda.synchronize()
    a._keep.pop("ingest_src", None)
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    assert a._ingest_seqs(th) == C
    extra = torch.cuda.max_memory_allocated() - before
    if 2 * C > 64:
        assert extra < th.numel() * 2 // n_seq, extra
    for s in range(n_seq):
        for (ka, va), (kb, vb) in zip(a.cache_tensors(s), b.cache_tensors(s)):
            assert torch.equal(ka[:, :C], kb[:, :C]) and torch.equal(va[:, :, :C], vb[:, :, :C])
