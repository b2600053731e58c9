"""Device mip chains against the host generator's, where the fused levels can go
wrong: sides around the 64-texel tile and the four-texel lane, odd sides at every
level, one axis kept from the start or from some level on, more levels than one
launch makes, and sources at odd byte addresses."""
import ctypes

import numpy as np
import pytest

import astc_encoder_amd as astc
from astc_encoder_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def enc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    e = astc.Encoder(0)
    yield e
    e.close()


@pytest.mark.parametrize("channels", [2, 3, 4])
@pytest.mark.parametrize("w,h", [(8, 8), (9, 7), (7, 9), (15, 64), (64, 64), (63, 65), (129, 127), (130, 11), (1, 300),
                                 (1027, 3), (5, 8200), (771, 513), (4099, 130)])
def test_mip_chain_edges(enc, channels, w, h):
    rng = np.random.default_rng(w * 7919 + h * 31 + channels)
    img = rng.integers(0, 256, size=(h, w, channels), dtype=np.uint8)
    want = synth.mip_chain(img)
    for offset in (0, 1):
        flat = torch.empty(img.size + 1, dtype=torch.uint8, device="cuda")
        base = flat[offset:offset + img.size].view(h, w, channels)
        base.copy_(torch.from_numpy(img))
        got = enc.mip_chain(base)
        assert got[0] is base and len(got) == len(want)
        for l, (g, x) in enumerate(zip(got, want)):
            np.testing.assert_array_equal(g.cpu().numpy(), x, err_msg=f"level {l}, offset {offset}")
        np.testing.assert_array_equal(enc.downsample(base).cpu().numpy(), want[1])


def test_mip_chain_writes_its_levels_only(enc):
    """Each level between guard bytes, for a ragged three-channel chain."""
    img = synth.sinusoid_rgb8(3, 203, 117)
    want = synth.mip_chain(img)[1:]
    base = torch.from_numpy(img).cuda()
    guard = 64
    bufs = [torch.full((x.size + 2 * guard,), 0xA5, dtype=torch.uint8, device="cuda") for x in want]
    desc = astc.make_desc(203, 117, astc.FMT_RGB8, 4, 0)
    ptrs = (ctypes.c_void_p * len(bufs))(*(b.data_ptr() + guard for b in bufs))
    stream = torch.cuda.current_stream().cuda_stream
    call = lambda n: astc.lib().astc_mip_chain(enc.handle, ctypes.byref(desc), base.data_ptr(), ptrs, n, stream)
    assert call(len(want)) == 0
    for b, x in zip(bufs, want):
        g = b.cpu().numpy()
        np.testing.assert_array_equal(g[guard:-guard].reshape(x.shape), x)
        assert (g[:guard] == 0xA5).all() and (g[-guard:] == 0xA5).all()
    assert call(0) == 0
    assert call(len(want) + 1) < 0
