"""astc_encode_batch_noalloc: the batched encode whose work list lives in the
library's fixed device array (no allocation per call).

Its blocks must equal those of the existing batched entry point
(astc_batch_create + astc_batch_launch, which allocates its work list) for
every image, bit for bit, on two calls in a row, the second with a smaller
batch (the array keeps the first call's contents; nothing of the first plan may
leak into the second).
"""
import ctypes

import numpy as np
import pytest

import astc_encoder_amd as astc
from astc_encoder_amd import synth
from astc_encoder_amd._capi import Tuning

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def enc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    e = astc.Encoder(0)
    yield e
    e.close()


def images_of(enc, seed, n, scale):
    """n textures of the mixed distribution (sides divided by `scale`) with their
    device mip chains, plus one max-accumulation image (a plain launch)."""
    out = []
    for mode, w, h, s in synth.draw_texture_specs(seed, n):
        gen, dim, flags, _ = synth.MODES[mode]
        base = torch.from_numpy(gen(s, max(4, w // scale), max(4, h // scale))).cuda()
        out += [(lvl, dim, flags) for lvl in enc.mip_chain(base)]
    img = torch.from_numpy(synth.noise_rgba8(seed + 7, 70, 45)).cuda()
    out.append((img, 6, astc.FLAG_ALPHA | astc.FLAG_MAX_ACCUMULATION))
    return out


def sentinel_outputs(images):
    outs = []
    for tex, dim, flags in images:
        h, w, c = tex.shape
        nb = astc.output_size(astc.make_desc(w, h, {4: 0, 3: 1, 2: 2}[c], dim, flags)) // 16
        outs.append(torch.full((nb, 16), 0xA5, dtype=torch.uint8, device="cuda"))
    return outs


def batch_reference(enc, images):
    b = astc.Batch(enc, images)
    b.set_tuning(4, 2, 1, 0)
    for o in b.outputs:
        o.fill_(0x5A)
    b.launch()
    torch.cuda.synchronize()
    ref = [o.cpu().numpy() for o in b.outputs]
    b.close()
    return ref


def test_noalloc_equals_batch_on_two_calls_second_smaller(enc):
    first = images_of(enc, 3, 24, 8)
    second = images_of(enc, 4, 6, 16)
    assert len(second) < len(first)
    want1, want2 = batch_reference(enc, first), batch_reference(enc, second)
    out1, out2 = sentinel_outputs(first), sentinel_outputs(second)
    print(f"no-alloc: {len(first)} then {len(second)} images", flush=True)
    enc.encode_batch_noalloc(first, out1)
    enc.encode_batch_noalloc(second, out2, tuning=(2, 1, 0, 2))
    torch.cuda.synchronize()
    for i, (o, w) in enumerate(zip(out1, want1)):
        np.testing.assert_array_equal(o.cpu().numpy(), w, err_msg=f"first call, image {i}")
    for i, (o, w) in enumerate(zip(out2, want2)):
        np.testing.assert_array_equal(o.cpu().numpy(), w, err_msg=f"second call, image {i}")


def test_noalloc_repeated_calls_on_one_stream(enc):
    images = images_of(enc, 5, 8, 8)
    want = batch_reference(enc, images)
    outs = sentinel_outputs(images)
    for _ in range(3):
        for o in outs:
            o.fill_(0xA5)
        enc.encode_batch_noalloc(images, outs, tuning=(8, 2, 1))
    torch.cuda.synchronize()
    for i, (o, w) in enumerate(zip(outs, want)):
        np.testing.assert_array_equal(o.cpu().numpy(), w, err_msg=f"image {i}")


@pytest.mark.parametrize("first", [True, False])
def test_a_captured_call_replays_its_own_images(enc, first):
    """A graph of one call, replayed between eager calls with other lists (longer and
    shorter) in the same array: every replay encodes the captured call's images.
    first: the captured call is the context's first."""
    images, longer, shorter = images_of(enc, 3, 24, 8), images_of(enc, 4, 40, 8), images_of(enc, 5, 2, 16)
    want, want_longer, want_shorter = (batch_reference(enc, x) for x in (images, longer, shorter))
    outs, outs_longer, outs_shorter = (sentinel_outputs(x) for x in (images, longer, shorter))
    own = astc.Encoder(0)
    if not first:
        own.encode_batch_noalloc(longer, outs_longer)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        own.encode_batch_noalloc(images, outs)
    for rep, (between, got, known) in enumerate([(longer, outs_longer, want_longer), (shorter, outs_shorter, want_shorter),
                                                 (longer, outs_longer, want_longer)]):
        for o in outs:
            o.fill_(0xA5)
        graph.replay()
        torch.cuda.synchronize()
        for i, (o, w) in enumerate(zip(outs, want)):
            np.testing.assert_array_equal(o.cpu().numpy(), w, err_msg=f"replay {rep}, image {i}")
        for o in got:
            o.fill_(0xA5)
        own.encode_batch_noalloc(between, got)
        torch.cuda.synchronize()
        for i, (o, w) in enumerate(zip(got, known)):
            np.testing.assert_array_equal(o.cpu().numpy(), w, err_msg=f"eager call {rep}, image {i}")
    del graph
    own.close()


def test_noalloc_refuses_what_exceeds_its_limits(enc):
    tex = torch.zeros((4, 4, 4), dtype=torch.uint8, device="cuda")
    out = torch.zeros((1, 16), dtype=torch.uint8, device="cuda")
    with pytest.raises(astc.AstcError, match="maximum"):
        enc.encode_batch_noalloc([(tex, 4, 0)] * 8193, [out] * 8193)
    d = (astc.ImageDesc * 1)(astc.make_desc(4, 4, astc.FMT_RGBA8, 4, 0))
    s = (ctypes.c_void_p * 1)(tex.data_ptr())
    o = (ctypes.c_void_p * 1)(out.data_ptr())
    rc = astc.lib().astc_encode_batch_noalloc(enc.handle, d, s, o, 1, ctypes.byref(Tuning(4, 2, 1, 1)), None)
    assert rc == -1 and b"split_modes" in astc.lib().astc_last_error()
    torch.cuda.synchronize()
