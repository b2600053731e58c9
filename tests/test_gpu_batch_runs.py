"""Batch work lists at their edges: one run of items or several, packs of one,
kMaxSegs and one more images, images one block below, at and above the 256 blocks
from which an image gets items of its own, the last item cut short, and the same
list through the allocation-free entry point.  Every image equals its plain encode."""
import numpy as np
import pytest

import astc_encoder_amd as astc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (channels, block size, flags): 6x6, four-channel 4x4, 4x4 RGB8 tiles, normal maps
KINDS = {"6": (4, 6, astc.FLAG_ALPHA | astc.FLAG_SRGB), "6r": (3, 6, astc.FLAG_SRGB), "4": (4, 4, astc.FLAG_ALPHA),
         "4s": (4, 4, astc.FLAG_SRGB), "r": (3, 4, 0), "rs": (3, 4, astc.FLAG_SRGB), "n": (2, 4, astc.FLAG_NORMAL)}
# blocks across and down of each image
PACKS = {"one": [(3, 2)], "sixteen": [(2, 1 + i % 3) for i in range(16)], "seventeen": [(1, 1)] * 17,
         "edges": [(15, 17), (16, 16), (257, 1), (1, 256), (17, 15), (51, 5), (1, 1)],
         "long": [(64, 100), (5, 300), (31, 7)]}


@pytest.fixture(scope="module")
def enc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    e = astc.Encoder(0)
    yield e
    e.close()


@pytest.mark.parametrize("pack", list(PACKS))
@pytest.mark.parametrize("kinds", ["6", "4", "r", "n", "6 n", "4 rs", "6r 4s", "6 6r 4 4s r rs n"])
def test_runs_and_packs(enc, kinds, pack):
    rng = np.random.default_rng(len(kinds) * 100 + len(pack))
    images = []
    for kind in kinds.split():
        c, dim, flags = KINDS[kind]
        for bw, bh in PACKS[pack]:
            cut = 0 if kind in ("r", "rs") else int(rng.integers(0, dim))
            w, h = bw * dim - cut, bh * dim
            images.append((torch.from_numpy(rng.integers(0, 256, size=(h, w, c), dtype=np.uint8)).cuda(), dim, flags))
    want = [enc.encode(t, d, f) for t, d, f in images]
    b = astc.Batch(enc, images)
    for tuning in ((4, 2, 1, 1, 1), (1, 1, 0, 0, 2), (8, 1, 1, 0, 1)):
        b.set_tuning(*tuning)
        for o in b.outputs:
            o.fill_(0xA5)
        b.launch()
        for i, (o, x) in enumerate(zip(b.outputs, want)):
            assert torch.equal(o, x), f"{tuning}: image {i}"
    b.close()
    outs = [torch.full_like(x, 0xA5) for x in want]
    enc.encode_batch_noalloc(images, outs)
    for i, (o, x) in enumerate(zip(outs, want)):
        assert torch.equal(o, x), f"no-alloc: image {i}"
