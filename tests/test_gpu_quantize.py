"""The quantiser's register and two-pass kernels bit-exact against the oracle at the edges of
their row lengths, with quotients at and next to halves and scales out of the reciprocal's
range."""

import numpy as np
import pytest

from mirror_sd_amd.config import workload
from oracle import dflash_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def quantizer():
    from mirror_sd_amd.dflash import DFlashDraftModel
    return DFlashDraftModel(workload("tiny").cfg, max_ctx=64)


@pytest.mark.parametrize("ic", [4, 1020, 4096, 4100, 8192, 12288, 12292, 20480, 20484, 4098])
def test_quantizer_row_lengths(quantizer, ic):
    rng = np.random.default_rng(ic)
    w = (rng.standard_normal((9, ic)) * 0.02).astype(np.float32)
    w[1] = 0.0
    w[2, :] = (rng.integers(-254, 255, ic) / 2).astype(np.float32)   # quotients at exact halves
    w[2, ic // 2] = 127.0
    w[3] *= np.float32(2.0 ** -113)   # a scale below 2^-100
    w[4] *= np.float32(2.0 ** 126)
    # quotients a few ulp either side of a half: the multiply alone would misround some
    half = (rng.integers(-126, 126, ic) + np.float32(0.5)).astype(np.float32)
    sc = np.float32(0.7310585975646973)
    w[5] = np.nextafter(half * sc, np.where(rng.random(ic) < 0.5, -np.inf, np.inf).astype(np.float32))
    w[5, 0] = np.float32(127.0) * sc
    q_ref, s_ref = O.quantize_w8(w)
    q, s = quantizer.quantize_w8(torch.from_numpy(w))
    np.testing.assert_array_equal(q.cpu().numpy(), q_ref)
    np.testing.assert_array_equal(s.cpu().numpy().view(np.uint16), s_ref.view(np.uint16))
