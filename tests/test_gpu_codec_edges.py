"""-m gpu: residual 1x1 contractions one behind the other (launch_gemm_chain): what a contraction writes for the one behind it is what that one reads - two planes, three, or f32
where the kernel in front writes another number of planes (96 .. 192 channels: f32; 224 .. 384: three planes behind a kernel that writes two; 768: two) - against float64."""
import ctypes as C

import numpy as np
import pytest

from mlx_audio_swift_amd import _lib
from mlx_audio_swift_amd.generation import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels, batch, columns", [(96, 2, 200), (192, 1, 130), (224, 1, 65), (256, 2, 129), (384, 1, 300), (768, 1, 130)])
def test_chain(channels, batch, columns):
    n, rng = 4, np.random.default_rng(channels)
    x = rng.standard_normal((batch, channels, columns)).astype(np.float32)
    wt = (rng.standard_normal((n, channels, channels)) / np.sqrt(channels)).astype(np.float32)
    bias = rng.standard_normal((n, channels)).astype(np.float32)
    alpha = rng.uniform(0.5, 1.5, channels).astype(np.float32)
    ralpha = (1.0 / alpha).astype(np.float32)
    got = np.empty_like(x)
    check(_lib.lib().mis_debug_codec_chain(0, n, channels, batch, columns, *(a.ctypes.data_as(C.c_void_p) for a in (x, wt, bias, alpha, ralpha, got))))
    ref = x.astype(np.float64)
    for i in range(n):
        s = ref + ralpha[:, None].astype(np.float64) * np.sin(alpha[:, None] * ref) ** 2
        ref = ref + np.einsum("kn,bkt->bnt", wt[i].astype(np.float64), s) + bias[i][:, None]
    # an operand of two planes keeps 16 bits (2^-17 of a value, halved in the mean over K), of three and f32 all of them; sine to 1e-6
    tol = 2e-5 if channels == 768 else 2e-6
    assert np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2)) <= tol
