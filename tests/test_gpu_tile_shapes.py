"""Prompt-sized ingests through every tile shape of the K|V product and through split and whole
fc products, at ragged row counts, against float64.  The cached rows carry three fp16 roundings
of normed values (the fc Linear, its norm, the k / v Linear; K one more through its norm and
one through the rotation): at most 5 * 2^-11 of each row's 2-norm."""

import pytest

from mirror_sd_amd import _lib, synth
from mirror_sd_amd.config import DFlashConfig
from parity_util import torch_tensors

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

H, NKV, NF = 1024, 8, 5


@pytest.fixture(scope="module")
def model():
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = DFlashConfig(hidden_size=H, num_hidden_layers=2, intermediate_size=512,
                       num_attention_heads=8, num_key_value_heads=NKV, head_dim=128,
                       vocab_size=512, block_size=8, target_layer_ids=[0, 1, 2, 3, 4],
                       num_target_layers=6)
    t = torch_tensors(synth.make_weights_numpy(cfg, seed=11), "cuda")
    m = DFlashDraftModel(cfg, max_ctx=2300)
    m.load_weights(t)
    yield cfg, t, m
    m.close()


def _rms(x, g, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * g.double()


def _lin(m, x, w):
    q, s = m.quantize_w8(w.float())
    return (x @ q.double().t()) * s.double()


def _check(model, th, slots=None, keep=None):
    """The cached rows of th's rows (those in ``keep``, at cache rows ``slots``)."""
    cfg, t, m = model
    rows = th.shape[0]
    keep = torch.arange(rows, device="cuda") if keep is None else keep
    slots = keep if slots is None else slots
    eps = cfg.rms_norm_eps
    h = _rms(th.double() @ t["fc.weight"].double().t(), t["hidden_norm.weight"], eps)
    f = cfg.rope_theta ** (-torch.arange(64, dtype=torch.float64, device="cuda") / 64)
    a = torch.arange(rows, dtype=torch.float64, device="cuda")[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    for i, (k, vt) in enumerate(m.cache_tensors(0)):
        p = f"layers.{i}.self_attn."
        kr = _rms(_lin(m, h, t[p + "k_proj.weight"]).reshape(rows, NKV, 128), t[p + "k_norm.weight"], eps)
        kr = torch.cat([kr[..., :64] * c - kr[..., 64:] * s, kr[..., 64:] * c + kr[..., :64] * s], -1)
        vr = _lin(m, h, t[p + "v_proj.weight"]).reshape(rows, NKV, 128)
        for got, want in ((k[:, slots].transpose(0, 1), kr[keep]),
                          (vt[:, :, slots].permute(2, 0, 1), vr[keep])):
            err = (got.double() - want).norm(dim=(1, 2)) / want.norm(dim=(1, 2))   # every row
            assert float(err.max()) <= 5 * 2.0 ** -11, (rows, i, float(err.max()))


def _rows(n):
    g = torch.Generator().manual_seed(n)
    return torch.randn((n, NF * H), generator=g).to(torch.float16).cuda()


@pytest.mark.parametrize("rows", [65, 129, 257, 600, 1100, 2100])
def test_ingest_rows(model, rows):
    th = _rows(rows)
    model[2].ingest_seq(0, th)
    _check(model, th)


@pytest.mark.parametrize("first,rows", [(3, 70), (4, 131), (1, 200)])
def test_append_at_any_row(model, first, rows):
    """V columns at cache rows that are and are not a multiple of four."""
    th = _rows(first + rows)
    model[2].ingest_seq(0, th[:first])
    model[2].ingest_seq(0, th[first:], reset=False)
    _check(model, th)


@pytest.mark.parametrize("first,rows", [(3, 150), (5, 97), (30, 70)])
def test_append_through_window(model, first, rows):
    """The same through a ring of 90 rows behind 5 sink rows (wraps inside the launch)."""
    m = model[2]
    sink, window = 5, 90
    m.make_cache(sink, window)
    th = _rows(first + rows)
    m.ingest_seq(0, th[:first])
    m.ingest_seq(0, th[first:], reset=False)
    n = first + rows
    keep = [r for r in range(n) if r < sink or r >= n - window]
    slots = m._cache_rows()
    m.make_cache(0, 0)
    assert len(keep) == slots.numel()
    _check(model, th, slots, torch.tensor(keep, device="cuda"))


@pytest.mark.parametrize("rows", [70, 131])
def test_wide_hidden_size(rows):
    """A hidden size above 5120 that is no multiple of 512 (the fc norm's larger register budget,
    its last step partly past the row)."""
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = DFlashConfig(hidden_size=5248, num_hidden_layers=1, intermediate_size=512,
                       num_attention_heads=NKV, num_key_value_heads=NKV, head_dim=128,
                       vocab_size=512, block_size=8, target_layer_ids=[1], num_target_layers=6)
    t = torch_tensors(synth.make_weights_numpy(cfg, seed=12), "cuda")
    m = DFlashDraftModel(cfg, max_ctx=rows)
    m.load_weights(t)
    g = torch.Generator().manual_seed(rows)
    th = torch.randn((rows, 5248), generator=g).to(torch.float16).cuda()
    m.ingest_seq(0, th)
    _check((cfg, t, m), th)
    m.close()


def _small(heads, kv, layers, F, **sizes):
    from mirror_sd_amd.dflash import DFlashDraftModel
    cfg = DFlashConfig(hidden_size=H, num_hidden_layers=layers, intermediate_size=F,
                       num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                       vocab_size=512, block_size=8, target_layer_ids=[0, 1, 2, 3, 4],
                       num_target_layers=6)
    m = DFlashDraftModel(cfg, **sizes)
    m.load_weights(torch_tensors(synth.make_weights_numpy(cfg, seed=11), "cuda"))
    return m


@pytest.mark.parametrize("rows", [65, 100, 257, 600])
def test_rows_do_not_depend_on_the_models_size(rows):
    """A prompt's cached rows are the same bits whatever number of context rows and layers the
    model was made for (the fc's split over K is a rule on the product alone)."""
    th, got = _rows(rows), []
    for layers, ctx in ((1, rows), (1, 4096), (3, rows)):
        m = _small(4, 4, layers, 512, max_ctx=ctx)
        m.ingest_seq(0, th)
        k, vt = m.cache_tensors(0)[0]
        got.append((k[:, :rows].clone(), vt[:, :, :rows].clone()))
        torch.cuda.synchronize()
        m.close()
    for k, vt in got[1:]:
        assert torch.equal(k, got[0][0]) and torch.equal(vt, got[0][1]), rows


@pytest.mark.parametrize("n_seq,block", [(2, 34), (2, 48)])
def test_stacked_block_does_not_depend_on_max_seqs(n_seq, block):
    """A stacked block's hidden states and logits are the same bits whatever number of sequences
    the model was made for (68 rows split the down product over K 16 ways, and the lm_head of
    512 columns where no ids are asked for).  Logits: fp32 sums of 1024 products in another
    order, 1024 * 2^-24 of their 2-norm at most."""
    th, got = _rows(40), []
    ids = (torch.arange(n_seq * block, dtype=torch.int32) % 512).reshape(n_seq, block).cuda()
    for seqs in (n_seq, 8):
        m = _small(4, 2, 1, 3584, max_ctx=40, max_block=48, max_seqs=seqs)
        for s in range(n_seq):
            m.ingest_seq(s, th)
        _, logits, hidden = m.draft_batch(ids=ids, return_logits=True, return_hidden=True)
        alone = torch.empty_like(logits)   # without ids
        _lib.check(m._L.dfl_draft_batch(m._ctx, n_seq, None, ids.data_ptr(), block, None, None,
                                        alone.data_ptr(), None, _lib.stream_handle()), "logits")
        got.append((hidden.clone(), logits.clone(), alone))
        torch.cuda.synchronize()
        m.close()
    for a, b in zip(*got):
        assert torch.equal(a, b), (n_seq, block)
    _, logits, alone = got[0]
    assert float((logits - alone).norm()) <= 1024 * 2.0 ** -24 * float(logits.norm())
