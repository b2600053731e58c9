"""Batch work lists at their edges: one run of items or several, packs of one,
kMaxSegs and one more images, images one block below, at and above the 256 blocks
from which an image gets items of its own, the last item cut short, and the same
list through the allocation-free entry point; and images large enough that a work
item is several steps.  Every image equals its plain encode."""
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


@pytest.mark.parametrize("kind", ["6", "6r", "6n", "4", "r", "rs", "n"])
@pytest.mark.parametrize("tuning,most", [((8, 2, 1, 1, 1), 8), ((8, 2, 0, 0, 2), 8), ((2, 2, 1, 0, 1), 2), ((8, 1, 0, 0, 1), 8)])
def test_several_steps_an_item(enc, kind, tuning, most):
    """An image of 1100 x 800 blocks (one tile repeated, whose blocks are known) beside
    small ones: at 256 blocks a step and two to five workgroups resident on each of 256
    compute units, chunks of three steps or more where the tuning lets them."""
    c, dim, flags = KINDS.get(kind) or (2, 6, astc.FLAG_NORMAL)
    rng = np.random.default_rng(dim + c)
    tile = torch.from_numpy(rng.integers(0, 256, size=(10 * dim, 100 * dim, c), dtype=np.uint8)).cuda()
    small = [(tile[:dim * k, :dim * 7].contiguous(), dim, flags) for k in (1, 3)]
    images = [(tile.repeat(80, 11, 1), dim, flags)] + small
    want = [enc.encode(tile, dim, flags).view(10, 100, 16).repeat(80, 11, 1).view(-1, 16)]
    want += [enc.encode(*x) for x in small]
    b = astc.Batch(enc, images)
    b.set_tuning(*tuning)
    resident = 1 if tuning[1] == 1 else {6: 3 if tuning[4] == 2 else 2, 4: 4 if c == 4 else 5}[dim]
    steps = min(most, -(-(1100 * 800 + 28) // (256 * 256 * resident)))
    assert steps >= 2 and b.info()["items"] == -(-1100 * 800 // (256 * steps)) + 1
    for o in b.outputs:
        o.fill_(0xA5)
    b.launch()
    for i, (o, x) in enumerate(zip(b.outputs, want)):
        assert torch.equal(o, x), f"image {i}"
    b.close()
    outs = [torch.full_like(x, 0xA5) for x in want]
    enc.encode_batch_noalloc(images, outs, tuning=(tuning[0], tuning[1], tuning[2], tuning[4]))
    for i, (o, x) in enumerate(zip(outs, want)):
        assert torch.equal(o, x), f"no-alloc: image {i}"
