"""The soft anchor's per-wave top-k lists at vocabulary sizes around a wave's slice and a scan
pass, with ties and NaN, into aligned and unaligned outputs (one fp16 step, as in
test_gpu_split.py: an fp32 sum rounded once)."""

import numpy as np
import pytest

from mirror_sd_amd import _lib
from oracle import dflash_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("V", [8, 255, 257, 2049, 163840, 163841, 400003])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_anchor_lists(V, dtype):
    H, k, dt = 64, min(8, V), getattr(torch, dtype)
    rng = np.random.default_rng(V)
    E = rng.normal(0, 0.02, (V, H)).astype(np.float16)
    lg = torch.from_numpy((rng.normal(0, 3, V)).astype(np.float32)).to(dt)
    lg[V // 2] = float("nan")
    lg[rng.integers(0, V, 5)] = 11.0   # ties across lists: the lower ids win
    lg[V - 1] = lg[0] = 11.0
    L, Ed, lgd = _lib.load(), torch.from_numpy(E).cuda(), lg.cuda()
    ids = torch.zeros(2, dtype=torch.int32, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    want = O.soft_anchor(E, lg.float().numpy(), top_k=k).astype(np.float64)
    buf = torch.zeros(2 * H + 8, dtype=torch.float16, device="cuda")
    for off in (0, 1):   # 16-byte rows, then element-wise rows
        out = buf[off:off + 2 * H]
        _lib.check(L.dfl_embed_block_noalloc(
            ids.data_ptr(), 2, Ed.data_ptr(), V, H, lgd.data_ptr(),
            {"float32": 0, "bfloat16": 2}[dtype], V, k, out.data_ptr(), err.data_ptr(),
            _lib.stream_handle()), "dfl_embed_block_noalloc")
        got = out.reshape(2, H).cpu().numpy()
        np.testing.assert_array_equal(got[1].view(np.uint16), E[0].view(np.uint16))
        step = np.spacing(np.maximum(np.abs(want), 2.0 ** -14).astype(np.float16)).astype(np.float64)
        assert (np.abs(got[0] - want) <= step).all()
    assert int(err.item()) == 0
