"""Sharing a plain launch's steps out over its workgroups: sizes with fewer steps than
resident workgroups, just as many, one more, a last step of one block, several steps
a workgroup with and without a longer one, and more than the consecutive order takes;
every lane count and texel form.  The image is one tile repeated, whose blocks are known."""
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


# blocks across and down; 512 (one lane), 768 (two lanes, packed) and 1280 workgroups
# are resident with 256 compute units, a step being 256 or 128 blocks
@pytest.mark.parametrize("bw,bh", [(256, 512), (257, 510), (131073, 1), (256, 769), (1000, 265), (640, 616), (1000, 600),
                                   (1366, 683)])
@pytest.mark.parametrize("tuning", [None, (1, 1, 0), (1, 8, 1, 1), (2, 4, 1), (1, 2, 0, 0, 1)])
def test_every_block_is_encoded_once(enc, bw, bh, tuning):
    rng = np.random.default_rng(bw + bh)
    tile = torch.from_numpy(rng.integers(0, 256, size=(60, 600, 4), dtype=np.uint8)).cuda()
    img = tile.repeat(-(-bh // 10), -(-bw // 100), 1)[:bh * 6, :bw * 6].contiguous()
    # the image repeats every 100 blocks across and 10 down: so do its blocks
    want = enc.encode(tile, 6, astc.FLAG_ALPHA, tuning=(1, 1, 0)).view(10, 100, 16)
    want = want.repeat(-(-bh // 10), -(-bw // 100), 1)[:bh, :bw]
    out = torch.full((bw * bh, 16), 0xA5, dtype=torch.uint8, device="cuda")
    enc.encode(img, 6, astc.FLAG_ALPHA, out=out, tuning=tuning)
    assert torch.equal(out.view(bh, bw, 16), want)
