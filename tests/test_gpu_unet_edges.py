"""GPU: the U-Net's weight and bias gradients at the edges of their tiles (32
columns by 8 or 16 rows, at full, half and quarter resolution), its forward
pass at the edges of strips, its minibatches.

The loss is made of few pixels: the target is the network's own output except
at the corners and on both sides of tile edges, 100 away, so that a pixel left
out or counted twice changes the gradients by far more than the tolerance, the
one test_gpu_unet.py has for BF16 storage (8% of a layer's norm).  With so few
pixels a ReLU whose sign BF16 storage changes counts for far more than in an
average over all of them, so the oracle rounds to BF16 where the network stores
a tensor.  The difference of the two sides' outputs elsewhere, of order 1e-2 on each of at most
9000 pixels, adds at most sqrt(9000) 1e-2 / (100 sqrt(9)) = 0.3%.  And the
gradients of four samples are those of the samples one by one: the loss's
1/(number of pixels) differs by a power of two, so every rounding to BF16 is the
same and only the order of FP32 sums differs (2e-5 of a layer's norm)."""
import numpy as np
import pytest

import tealeaf_hip as T
import unet_ref as U
from tealeaf_hip import decks, unet
from test_gpu_unet import bf16

pytestmark = pytest.mark.gpu


@pytest.fixture
def bf16_oracle(monkeypatch):
    conv, conv_back, pool, up_back = U.conv, U.conv_back, U.pool, U.up_back

    def back(x, w, dz):
        dx, dw, db = conv_back(x, w, bf16(dz))
        return bf16(dx), dw, db

    monkeypatch.setattr(U, "conv", lambda x, w, b: bf16(conv(x, w, b)))
    monkeypatch.setattr(U, "conv_back", back)
    monkeypatch.setattr(U, "pool", lambda x: bf16(pool(x)))
    monkeypatch.setattr(U, "up_back", lambda d: bf16(up_back(d)))


@pytest.fixture(scope="module")
def chunk():
    return T.initialiseapp(T.Settings.from_text(decks.reference_deck(16, 1)))


def _layers(g):
    o = 0
    for ci, _, co, _, _ in U.LAYERS:
        n = 9 * ci * co + co
        yield (ci, co), g[o:o + n]
        o += n


def _case(chunk, B, H, W):
    rng = np.random.default_rng(11)
    p = U.init_params(4).astype(np.float32)
    x = rng.standard_normal((B, H, W, 6)).astype(np.float32)
    unet.set_weights(chunk, p)
    target = np.array(unet.evaluate(chunk, x), dtype=np.float64).reshape(B, H, W)
    for y in {0, 7, 8, 15, 16, H - 1}:
        for xx in {0, 31, 32, W - 1}:
            if y < H and xx < W:
                target[:, y, xx] += 100.0
    return p, x, target


@pytest.mark.parametrize("shape", [(1, 8, 72), (3, 20, 36), (1, 68, 132), (2, 36, 4)])
def test_gradients_at_tile_edges(chunk, bf16_oracle, shape):
    print(f"case: unet gradients of edge pixels {shape}", flush=True)
    p, x, target = _case(chunk, *shape)
    _, loss, g = unet.evaluate(chunk, x, target)
    x16 = np.zeros(shape + (16,))
    x16[..., :6] = bf16(x)
    L, gref = U.loss_and_grads(bf16(p), x16, target)
    assert abs(loss - L) / L < 2e-2
    for (name, a), (_, b) in zip(_layers(g), _layers(gref)):
        assert np.linalg.norm(a - b) <= 8e-2 * np.linalg.norm(b) + 1e-6, name


@pytest.mark.parametrize("shape", [(1, 4, 4), (2, 36, 64), (1, 12, 516), (1, 100, 260)])
def test_forward_at_strip_edges(chunk, bf16_oracle, shape):
    """Strips of 64 columns (1, 2 or 4 of them to a block, at each of the three
    resolutions) and bands of 1 to 32 rows; test_gpu_unet.py's tolerance, on the
    whole output and on the columns and rows beside the edges."""
    print(f"case: unet forward {shape}", flush=True)
    p, x, _ = _case(chunk, *shape)
    out = np.asarray(unet.evaluate(chunk, x))
    x16 = np.zeros(shape + (16,))
    x16[..., :6] = bf16(x)
    ref, _ = U.forward(bf16(p), x16)
    cols = sorted({c for c in (0, 63, 64, 127, 128, 255, 256, shape[2] - 1) if c < shape[2]})
    rows = sorted({r for r in (0, 1, 2, 3, 31, 32, shape[1] - 1) if r < shape[1]})
    for a, b in ((out, ref), (out[:, :, cols], ref[:, :, cols]), (out[:, rows], ref[:, rows])):
        assert np.linalg.norm(a - b) < 2e-2 * np.linalg.norm(b)


@pytest.mark.parametrize("shape", [(4, 20, 36), (4, 64, 72)])
def test_gradients_of_a_batch_are_those_of_its_samples(chunk, shape):
    print(f"case: unet gradients of a batch {shape}", flush=True)
    _, x, target = _case(chunk, *shape)
    _, _, g = unet.evaluate(chunk, x, target)
    s = sum(unet.evaluate(chunk, x[b:b + 1], target[b:b + 1])[2].astype(np.float64) for b in range(4)) / 4
    for (name, a), (_, b) in zip(_layers(g), _layers(s)):
        assert np.linalg.norm(a - b) <= 2e-5 * np.linalg.norm(b), name


def test_batches_of_one_sample():
    """Minibatches are gathered 64 samples at a time: drawn from a dataset of
    one sample (the whole grid, with edges on all sides), a batch of any size
    has that sample's loss.  The 256-pixel sums are the same for each of its
    copies and are added in FP64, so only the scale's rounding (2^-24) differs."""
    print("case: minibatches of 1 to 130 copies of one sample", flush=True)
    s = T.Settings.from_text(decks.random_rect_deck(21, n=128, steps=1))
    c = T.initialiseapp(s)
    unet.record(c, capacity=1, crops_per_step=1)
    T.diffuse(c, s, 1)
    assert unet.dataset_size(c) == 1
    for kind in ("energy", "mse", "residual"):
        loss = [unet.train(c, steps=2, batch=b, lr=0.0, loss=kind) for b in (1, 3, 64, 65, 130)]
        assert np.all(np.isfinite(loss)) and np.min(loss) > 0.0
        np.testing.assert_allclose(loss, np.full_like(loss, loss[0][0]), rtol=1e-6)
