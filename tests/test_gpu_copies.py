"""The copy kernel behind the server and the allocation-free batch: many ranges in
one launch.  Requests of every size from one block up, more of them than one launch
takes, with sources at odd byte addresses and destinations at every one (those that
are not 16-byte aligned are copied out, others written in place), each with guard
bytes around its destination."""
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


@pytest.mark.parametrize("count,most", [(1, 8), (64, 40), (150, 300)])
def test_requests_of_every_size(enc, count, most):
    rng = np.random.default_rng(count)
    reqs, wants, dsts = [], [], []
    for i in range(count):
        c, dim = int(rng.integers(2, 5)), int(rng.choice([4, 6]))
        flags = astc.FLAG_NORMAL if c == 2 else astc.FLAG_ALPHA if c == 4 else 0
        w, h = (int(v) for v in rng.integers(1, most, 2))
        img = torch.from_numpy(rng.integers(0, 256, size=(h, w, c), dtype=np.uint8)).cuda()
        p = astc.PackedImages([img], dim, flags)
        shift = int(rng.integers(0, 4))
        moved = torch.empty(p.buffer.numel() + shift, dtype=torch.uint8, device="cuda")
        moved[shift:].copy_(p.buffer)
        p.buffer = moved[shift:]
        dst = torch.full((p.out_bytes + 48,), 0xA5, dtype=torch.uint8, device="cuda")
        at = 16 + (0 if i % 4 == 3 else int(rng.integers(1, 16)))
        reqs.append((p, 0.0, dst[at:]))
        dsts.append((dst, at))
        wants.append(enc.encode(img, dim, flags).cpu().numpy().reshape(-1))
    torch.cuda.synchronize()
    srv = astc.Server(enc, 64 << 20, max_inflight=2, max_batch_requests=100)
    srv.run_trace(reqs)
    srv.close()
    # several pieces of a range, and more ranges copied out than one launch takes
    if count == 150:
        assert max(len(w) for w in wants) > 2 * 32768 and sum(at > 16 for _, at in dsts[:100]) > 64
    for (dst, at), want in zip(dsts, wants):
        got, end = dst.cpu().numpy(), at + len(want)
        np.testing.assert_array_equal(got[at:end], want)
        assert (got[:at] == 0xA5).all() and (got[end:] == 0xA5).all()


@pytest.mark.parametrize("how,slots,per_batch", [("own source", 1, 6), ("another's source", 1, 6),
                                                 ("one destination", 1, 6), ("none", 1, 6), ("own source", 3, 2),
                                                 ("one destination", 3, 2), ("none", 3, 2)])
def test_overlapping_destinations(enc, how, slots, per_batch):
    """Destinations over sources of the same trace: every source of a batch is read
    before any of its blocks is written; requests with one destination leave the last
    one's blocks, in one batch or in several with three in flight."""
    rng = np.random.default_rng(5)
    imgs = [torch.from_numpy(rng.integers(0, 256, size=(96, 128, 4), dtype=np.uint8)).cuda() for _ in range(6)]
    packs = [astc.PackedImages([t], 4, astc.FLAG_ALPHA) for t in imgs]
    wants = [enc.encode(t, 4, astc.FLAG_ALPHA).view(-1) for t in imgs]
    n = packs[0].out_bytes
    dsts = [torch.empty(n, dtype=torch.uint8, device="cuda") for _ in imgs]
    if how == "own source":
        dsts = [p.buffer[:n] for p in packs]
    elif how == "another's source":
        dsts = [packs[(i + 1) % len(packs)].buffer[:n] for i in range(len(packs))]
    elif how == "one destination":
        dsts = [dsts[0]] * len(packs)
    torch.cuda.synchronize()
    srv = astc.Server(enc, 8 << 20, max_inflight=slots, max_batch_requests=per_batch)
    srv.run_trace([(p, 0.0, d) for p, d in zip(packs, dsts)])
    srv.close()
    for i, (d, want) in enumerate(zip(dsts, wants)):
        assert torch.equal(d, wants[-1] if how == "one destination" else want), i
