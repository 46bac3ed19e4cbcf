"""The decoding layer's one-launch weight casts: widths whose transposed tiles are cut on either side, 16-byte
rows or not, and a weight array that starts off the 16-byte grid."""
import numpy as np
import pytest
import torch

from conftest import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,d,H,ffn,shift", [
    (2, 9, 40, 1, 20, 0),         # the feed-forward half the library's by width; scalar tiles, cut on both sides
    (2, 9, 64, 1, 64, 0),         # plain casts, biases shorter than a block
    (40, 120, 200, 5, 328, 0),    # the library's by size; vector tiles, cut at 200 and 328
    (40, 120, 200, 5, 328, 1),    # the same from unaligned sources
    (6, 800, 1088, 17, 1088, 0),  # whole tiles
])
def test_decoding_layer_cast_edges(pkg, gpu, oracle, rng, B, S, d, H, ffn, shift):
    f = lambda *s: (0.03 * rng.standard_normal(s)).astype(np.float32)
    x = rng.standard_normal((B, S, d)).astype(np.float32)
    W = [f(d, 3 * d), f(d, d), f(d), f(d, ffn), f(ffn), f(ffn, d), f(d)]

    def place(w):
        flat = torch.empty(w.size + shift, device=gpu)
        flat[shift:] = torch.from_numpy(w.ravel()).to(gpu)
        return flat[shift:].view(*w.shape)

    dev = [place(w) for w in W]
    got = pkg.decoding_context_layer(to_dev(x, gpu), *dev, heads=H).cpu().numpy()
    rows = min(B, 2)  # sequences are independent of each other
    ref = oracle.decoding_context_layer(x[:rows], *W, heads=H)
    err = np.abs(got[:rows] - ref)
    assert np.all(err <= 2e-2 + 2e-2 * np.abs(ref)), err.max()
    again = pkg.decoding_context_layer(to_dev(x[-rows:], gpu), *dev, heads=H).cpu().numpy()  # (other kernels, by size)
    assert np.allclose(got[-rows:], again, rtol=2e-2, atol=2e-2)
