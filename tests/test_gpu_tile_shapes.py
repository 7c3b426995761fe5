"""Prompt-sized ingests through every tile shape of the K|V product and through split and whole
fc products, at ragged row counts, against float64.  The cached rows carry three fp16 roundings
of normed values (the fc Linear, its norm, the k / v Linear; K one more through its norm and
one through the rotation): at most 5 * 2^-11 of the 2-norm."""

import pytest

from mirror_sd_amd import synth
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


@pytest.mark.parametrize("rows", [65, 129, 257, 600, 1100, 2100])
def test_ingest_rows(model, rows):
    cfg, t, m = model
    g = torch.Generator().manual_seed(rows)
    th = torch.randn((rows, NF * H), generator=g).to(torch.float16).cuda()
    m.ingest_seq(0, th)
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
        for got, want in ((k[:, :rows].transpose(0, 1), kr), (vt[:, :, :rows].permute(2, 0, 1), vr)):
            err = float((got.double() - want).norm() / want.norm())
            assert err <= 5 * 2.0 ** -11, (rows, i, err)
