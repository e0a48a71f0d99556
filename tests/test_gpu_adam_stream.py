"""The training step's update kernel streams the SH arrays past the caches from 128 MB on
(parameters and moments, 36 sh_k bytes per Gaussian): every row must get the bits that the same
row gets in a call too small to stream."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = ((3,), (3,), (4,), (1,))


def _update(cuda, rows, K, degree, x):
    """One gs_preprocess_bwd_adam call on copies of some rows; the updated arrays."""
    import ctypes

    from jax_gs_amd import _lib

    p = [t[rows].clone() for t in x["params"]]
    mo = [t[rows].clone() for t in x["mu"] + x["nu"]]
    grec, active = x["grec"][rows].clone(), x["active"][rows].clone()
    n = p[0].shape[0]
    moments = (ctypes.c_void_p * 10)(*[t.data_ptr() for t in mo])
    lrs = (ctypes.c_double * 5)(1e-3, 5e-3, 1e-3, 5e-2, 2.5e-3)
    _lib.call("gs_preprocess_bwd_adam", _lib.stream_handle(cuda), n, K, degree, *[_lib.ptr(t) for t in p],
              _lib.ptr(x["w2c"]), 64, 48, 60.0, 60.0, 32.0, 24.0, _lib.ptr(grec), moments, lrs, 3, 0.9, 0.999, 1e-8,
              _lib.ptr(active), None, None, 60.0, 1.0, None, None, None)
    return p + mo


@pytest.mark.parametrize("K, degree, over", [(16, 3, 0), (16, 1, 1), (9, 2, 0), (5, 1, 130)])
def test_streamed_update_matches_small_calls(cuda, K, degree, over):
    n = -(-(128 << 20) // (36 * K)) + over  # the smallest n that streams, and a little more
    gen = torch.Generator(device=cuda).manual_seed(5)

    def randn(*s):
        return torch.randn(s, generator=gen, device=cuda)

    shapes = SHAPES + ((K, 3),)
    x = {"params": [randn(n, *s) for s in shapes], "mu": [0.1 * randn(n, *s) for s in shapes],
         "nu": [0.01 * randn(n, *s).square() for s in shapes], "grec": randn(n, 12),
         "active": (torch.rand(n, generator=gen, device=cuda) < 0.7).to(torch.uint8),
         "w2c": torch.eye(4, device=cuda)}
    x["params"][0][:, 2] += 4.0
    whole = _update(cuda, slice(0, n), K, degree, x)
    for a, b in ((0, 4097), (n // 2, n // 2 + 200), (n - 131, n)):
        part = _update(cuda, slice(a, b), K, degree, x)
        for w, q in zip(whole, part):
            np.testing.assert_array_equal(w[a:b].cpu().numpy(), q.cpu().numpy())
