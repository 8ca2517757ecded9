"""Row-layout attention (ck_attention) at every key split a wave can own: T from
64 to 512 (32 keys per wave up to 256, 64 above), both head widths, head counts
that do not fill an XCD, keys whose order matters (one key dominating each
query at a place of its own) -- against the oracle, at its f16 output bound."""
import numpy as np
import pytest

from oracle import model as OM
from test_gpu_kernels import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('hd', [64, 128])
@pytest.mark.parametrize('T,H', [(64, 1), (128, 3), (192, 2), (256, 5), (320, 1), (448, 3), (512, 2)])
@pytest.mark.parametrize('peaked', [False, True])
def test_attention_row_layout_key_order(gpu, T, H, hd, peaked):
    from chestnut import kernels as K
    rng = np.random.default_rng(T + H + hd)
    d = H * hd
    qkv = rng.standard_normal((T, 3 * d))
    if peaked:   # query t looks at key (37 t + 5) mod T: its output is that key's V row
        at = (37 * np.arange(T) + 5) % T
        qkv[:, :d] = 6.0 * qkv[at, d:2 * d]
    qkv = OM.f16r(qkv)
    out = host(K.attention(dev(gpu, qkv[:, :2 * d].astype(np.float16)),
                           dev(gpu, np.ascontiguousarray(qkv[:, 2 * d:].T).astype(np.float16)), H, hd)).astype(np.float64)
    ref = OM.attention(qkv, H, hd)
    assert np.max(np.abs(out - ref)) <= 2.0 ** -9 * np.max(np.abs(ref))
