"""The hybrid decoder's prompt mixers where their launches change shape: linear attention in one piece and in segments, softmax attention in tiles of
64 and of 128 query rows, keys of the pass and of the cache in one tile; against the plain implementation, as in test_hip_hybrid.py."""
import numpy as np
import pytest

from crabml_amd import synth_bifazen as sb
from crabml_amd import synth_hybrid as sh
from tests import test_hip_bifazen as bifazen
from tests.test_hip_hybrid import Model, close

pytestmark = pytest.mark.gpu

# decays that carry a state over a thousand rows, so that a segment that starts from the wrong one shows
LINEAR = sh.config(72, 99, [sh.layer(2, 1, 16, 24, 300, 3, 24, 40, 48, decay=[0.999, 0.99, 0.9]), sh.layer(2, 2, 8, 8, 40, 1, 72, 8, None, decay=[0.998])])
# heads between 64 and 128 wide: few tiles give two waves the same rows, eight tiles of 128 rows of 64 heads and more go to the larger tiles
FEW_HEADS = sh.config(64, 77, [sh.layer(4, 2, 104, 128, 256, 1, 8, 8, None), sh.layer(2, 1, 128, 72, 1000, 1, 8, 8, None)])
MANY_HEADS = sh.config(64, 77, [sh.layer(64, 2, 72, 80, 600, 1, 8, 8, None)])


@pytest.fixture(scope="module")
def linear(tmp_path_factory):
    return Model(LINEAR, tmp_path_factory.mktemp("linear"), seed=3)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("n", [127, 128, 129, 255, 256, 257, 320, 641, 1000])
def test_one_prompt(ca, hdev, linear, n, f32):
    r = linear.runner(ca, hdev, f32, seq_len=1100)
    t = linear.tokens(n + 3, seed=n)
    want = linear.oracle(t)
    s = r.open()
    close(r.step([(s, t[:n], list(range(n)))]), want[:n], f32)
    for i in range(n, n + 3):  # the state and the cache that it leaves
        close(r.step([(s, [t[i]], [0])]), want[i:i + 1], f32)


@pytest.mark.parametrize("f32", [True, False])
def test_portions_and_neighbours(ca, hdev, linear, f32):
    """a state to start from, with sequences of one block, of some and of many in the same pass; keys of the cache and the pass in one tile"""
    r = linear.runner(ca, hdev, f32, seq_len=1100)
    lens, cuts = [900, 70, 333], [100, 30, 45]
    prompts = [linear.tokens(n, seed=n) for n in lens]
    seqs = [r.open() for _ in lens]
    want = [linear.oracle(p) for p in prompts]
    r.step([(s, p[:c], [c - 1]) for s, p, c in zip(seqs, prompts, cuts)])
    got = r.step([(s, p[c:], list(range(len(p) - c))) for s, p, c in zip(seqs, prompts, cuts)])
    close(got, np.concatenate([w[c:] for w, c in zip(want, cuts)]), f32)


@pytest.mark.parametrize("heads,n", [("few", 51), ("few", 82), ("few", 83), ("few", 114), ("few", 115), ("few", 700), ("many", 895), ("many", 897), ("many", 946), ("many", 947), ("many", 1040)])
def test_query_tiles(ca, hdev, tmp_path, heads, n):
    m = Model(FEW_HEADS if heads == "few" else MANY_HEADS, tmp_path, seed=5)
    r = m.runner(ca, hdev, False, seq_len=1100)
    t = m.tokens(n, seed=n)
    s = r.open()
    got = [r.step([(s, t[:50], list(range(50)))]), r.step([(s, t[50:], list(range(n - 50)))])]
    close(np.concatenate(got), m.oracle(t), False)


# 64 heads: eight tiles of 128 rows and more go to the larger tiles -- with a latent key of up to 128 and of up to 192 columns, and in a window
LATENT_128 = sb.config(64, 77, [sb.latent(64, 72, 20, 80, 32, 300, None)])
LATENT_192 = sb.config(64, 77, [sb.latent(64, 120, 32, 104, 40, 1000, None)])
WINDOW = sb.config(64, 77, [sb.attention(64, 2, 72, 80, 200, None)])


@pytest.mark.parametrize("config", [LATENT_128, LATENT_192, WINDOW])
@pytest.mark.parametrize("n", [946, 947, 1075])
def test_query_tiles_of_latent_and_windowed_heads(ca, hdev, tmp_path, config, n):
    """896, 897 and 1025 rows behind 50 that are in the cache: seven, eight and nine tiles, the last one whole, of one row and of one row"""
    m = bifazen.Model(config, tmp_path, seed=6)
    r = m.runner(ca, hdev, False, seq_len=1100)
    t = m.tokens(n, seed=n)
    s = r.open()
    got = [r.step([(s, t[:50], list(range(50)))]), r.step([(s, t[50:], list(range(n - 50)))])]
    bifazen.close(np.concatenate(got), m.oracle(t), False)
