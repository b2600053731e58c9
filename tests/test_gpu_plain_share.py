"""Sharing a plain launch's steps out over its workgroups: sizes with fewer steps than
resident workgroups, just as many, one more, a last step of one block, several steps
a workgroup with and without a longer one, and more than the consecutive order takes;
every lane count and texel form, block size and channel class.  The image is one tile
repeated, whose blocks are known."""
import numpy as np
import pytest

import astc_encoder_amd as astc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def enc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    e = astc.Encoder(0)
    yield e
    e.close()


def repeated(enc, tile, dim, flags, bw, bh):
    """The image of bw x bh blocks that repeats a tile of 100 x 10 blocks, and its blocks."""
    img = tile.repeat(-(-bh // 10), -(-bw // 100), 1)[:bh * dim, :bw * dim].contiguous()
    want = enc.encode(tile, dim, flags, tuning=(1, 1, 0)).view(10, 100, 16)
    return img, want.repeat(-(-bh // 10), -(-bw // 100), 1)[:bh, :bw]


# blocks across and down; 6x6 encodes have 512 (one lane) or 768 workgroups (two lanes,
# packed) resident with 256 compute units, a step being 256 or 128 blocks
@pytest.mark.parametrize("bw,bh", [(256, 512), (257, 510), (131073, 1), (256, 769), (1000, 265), (640, 616), (1000, 600),
                                   (1366, 683)])
@pytest.mark.parametrize("tuning", [None, (1, 1, 0), (1, 8, 1, 1), (2, 4, 1), (1, 2, 0, 0, 1)])
def test_every_block_is_encoded_once(enc, bw, bh, tuning):
    rng = np.random.default_rng(bw + bh)
    tile = torch.from_numpy(rng.integers(0, 256, size=(60, 600, 4), dtype=np.uint8)).cuda()
    img, want = repeated(enc, tile, 6, astc.FLAG_ALPHA, bw, bh)
    out = torch.full((bw * bh, 16), 0xA5, dtype=torch.uint8, device="cuda")
    enc.encode(img, 6, astc.FLAG_ALPHA, out=out, tuning=tuning)
    assert torch.equal(out.view(bh, bw, 16), want)


# (channels, block size, flags, alpha): 4x4 encodes have 1024 workgroups resident,
# packed 1280.  Blocks: one, two and more than four steps a workgroup of the 4x4 forms
KINDS = {"rgb 6": (3, 6, 0, None), "rgb srgb 6": (3, 6, astc.FLAG_SRGB, None), "normal 6": (2, 6, astc.FLAG_NORMAL, None),
         "flat 6": (4, 6, astc.FLAG_ALPHA, "flat"), "search 6": (4, 6, astc.FLAG_ALPHA | astc.FLAG_MAX_ACCUMULATION, None),
         "rgba 4": (4, 4, astc.FLAG_ALPHA, None), "flat 4": (4, 4, astc.FLAG_SRGB, "flat"), "rgb 4": (3, 4, 0, None),
         "normal 4": (2, 4, astc.FLAG_NORMAL, None)}


@pytest.mark.parametrize("bw,bh", [(1000, 270), (1000, 600), (1366, 1000)])
@pytest.mark.parametrize("kind", list(KINDS))
def test_several_steps_of_every_class(enc, kind, bw, bh):
    channels, dim, flags, alpha = KINDS[kind]
    rng = np.random.default_rng(bw + bh)
    tile = rng.integers(0, 256, size=(10 * dim, 100 * dim, channels), dtype=np.uint8)
    if alpha == "flat":  # whole waves of opaque blocks, of others, and mixed ones
        tile[:5 * dim, :, 3] = 255
    img, want = repeated(enc, torch.from_numpy(tile).cuda(), dim, flags, bw, bh)
    if bh == 600:  # rows off their words: the other kind of row loads, several steps ahead
        moved = torch.empty(img.numel() + 1, dtype=torch.uint8, device="cuda")
        moved[1:].copy_(img.view(-1))
        img = moved[1:].view(img.shape)
    for tuning in (None, (1, 8, 0), (1, 8, 1), (1, 8, 0, 1), (1, 2, 1, 1), (2, 8, 1), (2, 8, 0), (1, 8, 0, 0, 1)):
        out = torch.full((bw * bh, 16), 0xA5, dtype=torch.uint8, device="cuda")
        enc.encode(img, dim, flags, out=out, tuning=tuning)
        assert torch.equal(out.view(bh, bw, 16), want), tuning
