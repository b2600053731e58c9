"""Sources whose rows begin at any byte: every format and block size at widths that
leave each remainder of four bytes, and at each source offset, plain in every form (a
packed-texel kernel holds the loads of aligned or of other rows) and in a batch, against
the oracle.
The source ends with its last texel, and the bytes around it are set to a value that
would show."""
import numpy as np
import pytest

import astc_encoder_amd as astc
from tests.oracle_ref import oracle_encode

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def enc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    e = astc.Encoder(0)
    yield e
    e.close()


@pytest.mark.parametrize("dim", [4, 6])
@pytest.mark.parametrize("channels,flags", [(3, 0), (3, astc.FLAG_SRGB), (2, astc.FLAG_NORMAL), (2, 0), (4, astc.FLAG_ALPHA),
                                            (3, astc.FLAG_NORMAL)])
@pytest.mark.parametrize("w,h", [(12, 12), (13, 18), (37, 11), (62, 24), (91, 30)])
def test_rows_at_any_byte(enc, dim, channels, flags, w, h):
    rng = np.random.default_rng(w * 131 + h * 7 + channels)
    img = rng.integers(0, 256, size=(h, w, channels), dtype=np.uint8)
    want = oracle_encode(img, dim, flags)
    for offset in range(4):
        flat = torch.full((img.size + offset + 4,), 0xA5, dtype=torch.uint8, device="cuda")
        src = flat[offset:offset + img.size].view(h, w, channels)
        src.copy_(torch.from_numpy(img))
        for tuning in (None, (1, 1, 0), (2, 1, 1), (1, 1, 0, 0, 1)):
            got = enc.encode(src, dim, flags, tuning=tuning).cpu().numpy()
            np.testing.assert_array_equal(got, want, err_msg=f"offset {offset} tuning {tuning}")
        b = astc.Batch(enc, [(src, dim, flags)])
        for lanes in (1, 2):
            b.set_tuning(4, 2, 1, 1, lanes)
            b.outputs[0].fill_(0xA5)
            b.launch()
            np.testing.assert_array_equal(b.outputs[0].cpu().numpy(), want, err_msg=f"offset {offset} batch {lanes}")
        b.close()
