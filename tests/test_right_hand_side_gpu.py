"""The transposed copy of a bf16 [K][N] right-hand side, in its 16-byte and its element-wise form, against float64."""
import numpy as np
import pytest

import test_kernels_gpu as T
from oracle import tile_oracle as E
from plaidml_amd import hipkernels as hk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('K,N', [(8, 4), (136, 68), (128, 64), (264, 1000), (40, 7), (4096, 260)])
def test_bf16_right_hand_side_turned(K, N, monkeypatch):
    """Every element has to arrive: ragged 64 x 128 tiles of the copy, rows that are no whole vectors."""
    hk.init(0)
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile('64x64'))  # (a tile that reads Bt)
    rng = np.random.default_rng(K)
    A, B = (E.round_bf16(rng.standard_normal(s).astype(np.float32)) for s in ((24, K), (K, N)))
    got = E.bf16_from_bits(T.run_gemm(T.bf16(A), T.bf16(B), hk.BF16, hk.BF16))
    # one rounding to bf16 of a sum of K products, itself summed in fp32
    np.testing.assert_allclose(got, A.astype(np.float64) @ B.astype(np.float64), rtol=2.0 ** -8, atol=2.0 ** -24 * K * np.sqrt(K) + 1e-6)
