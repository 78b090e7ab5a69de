"""bz_feed: a contiguous range and strided pieces out of pinned host memory, against the bytes themselves."""
import ctypes as C

import pytest
import torch

import blaze_hip as bz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("range_bytes,pieces", [
    (0, [(1, 1, 1, 1)]),                                      # the smallest piece
    (16, []),
    (16384 * 3 + 16, [(300, 26, 26, 890)]),                   # a workgroup's edge, odd rows in a wide tensor
    (1 << 20, [(2048, 128, 128, 1792), (7, 3, 5, 11)]),       # 16-byte units and single bytes in one launch
    (0, [(5, 8, 8, 24), (1025, 4, 4, 12), (0, 4, 4, 4), (513, 2, 2, 2), (1, 16384, 16384, 16384), (3, 48, 64, 80), (2, 12, 12, 12),
         (9, 1, 1, 2)]),                                      # every unit, an empty piece, as many pieces as a launch takes
])
def test_feed(range_bytes, pieces):
    gen = torch.Generator().manual_seed(range_bytes + len(pieces))

    def rand(n):
        return torch.randint(256, (max(n, 1), ), generator=gen, dtype=torch.uint8)

    src = rand(range_bytes).pin_memory()
    dst = torch.full((max(range_bytes, 1) + 16, ), 7, dtype=torch.uint8, device="cuda")
    rows = (bz.FeedRows * max(len(pieces), 1))()
    keep = []
    for i, (n, w, sp, dp) in enumerate(pieces):
        s = rand(n * sp).pin_memory()
        d = torch.full((n * dp + 16, ), 9, dtype=torch.uint8, device="cuda")
        keep.append((s, d))
        rows[i].src, rows[i].dst, rows[i].rows, rows[i].row_bytes, rows[i].src_pitch, rows[i].dst_pitch = s.data_ptr(), d.data_ptr(), n, w, sp, dp
    bz.check(bz.lib().bz_feed(src.data_ptr(), dst.data_ptr(), range_bytes, rows, len(pieces), bz._stream_ptr()))
    got = dst.cpu()
    assert torch.equal(got[:range_bytes], src[:range_bytes]) and bool((got[range_bytes:] == 7).all())
    for (n, w, sp, dp), (s, d) in zip(pieces, keep):
        want = torch.full((n * dp + 16, ), 9, dtype=torch.uint8)
        for r in range(n):
            want[r * dp:r * dp + w] = s[r * sp:r * sp + w]
        assert torch.equal(d.cpu(), want), (n, w, sp, dp)


@pytest.mark.parametrize("range_bytes,pieces", [
    (320 << 10, []),                                           # the most of which a lane asks for one unit at a time
    ((320 << 10) + 16, []),
    ((320 << 10) - 7 * 130, [(7, 130, 132, 140)]),             # the same with pieces
    ((320 << 10) - 7 * 130 + 16, [(7, 130, 132, 140)]),
    (384 << 10, []),                                           # two units, whole and partial workgroups
    ((384 << 10) + 16, []),
    ((384 << 10) - 7 * 130, [(7, 130, 132, 140)]),
    ((384 << 10) - 7 * 130 + 16, [(7, 130, 132, 140)]),
    (4096, [(257, 1, 1, 3), (2, 255, 256, 300), (256, 3, 4, 5)]),                       # pieces of a workgroup and one unit
    (400000, [(513, 1, 1, 3), (2, 511, 512, 600), (1, 512, 512, 512), (3001, 6, 6, 9)]),  # the same at two units a lane
    (0, [(1, 100000, 100000, 100000), (100000, 1, 2, 1), (40000, 7, 8, 7)]),             # rows longer than a workgroup, and shorter than a lane's stride
])
def test_feed_at_the_edges_of_its_two_sizes(range_bytes, pieces):
    test_feed(range_bytes // 16 * 16, pieces)


def test_feed_refuses():
    rows = (bz.FeedRows * 9)()
    buf = torch.zeros(64, dtype=torch.uint8).pin_memory()
    call = bz.lib().bz_feed
    p = buf.data_ptr()
    assert call(p, p, 24, rows, 0, None) == bz.EINVAL      # no multiple of 16 bytes
    assert call(p + 4, p, 16, rows, 0, None) == bz.EINVAL  # misaligned
    assert call(None, None, 0, rows, 9, None) == bz.EINVAL
    rows[0] = bz.FeedRows(p, p, 2, 8, 4, 8)                # rows that overlap
    assert call(None, None, 0, rows, 1, None) == bz.EINVAL
    assert C.sizeof(bz.FeedRows) == 48


def _pieces(spec, gen):
    """[(form, bytes)] -> (pieces, what lies at each destination before, what has to lie there after, what must stay alive)"""
    pieces, dsts, wants, keep = (bz.FeedPiece * max(len(spec), 1))(), [], [], []
    for i, (form, n) in enumerate(spec):
        dst = torch.full((n + 16, ), 7, dtype=torch.uint8, device="cuda")
        want = torch.full((n + 16, ), 7, dtype=torch.uint8)
        word = int(torch.randint(1 << 31, (1, ), generator=gen)) * 2 + 1
        if form == bz.FEED_SAME32:
            want[:n] = torch.tensor([word - (1 << 32) if word >> 31 else word] * (n // 4), dtype=torch.int32).view(torch.uint8)
            src = None
        else:
            src = torch.randint(256, ((n if form == bz.FEED_RAW else n // 2 + 15) // 16 * 16, ), generator=gen, dtype=torch.uint8).pin_memory()
            if form == bz.FEED_RAW:
                want[:n] = src
            else:
                want[:n].view(torch.int32).view(-1, 2).copy_(torch.stack([src[:n // 2].view(torch.int32), torch.zeros(n // 8, dtype=torch.int32)], 1))
        pieces[i] = bz.FeedPiece(src.data_ptr() if src is not None and n else None, dst.data_ptr(), n, form, word)
        dsts.append(dst)
        wants.append(want)
        keep.append(src)
    return pieces, dsts, wants, keep


RAW, LOW, SAME = 0, 1, 2


@pytest.mark.parametrize("spec", [
    [(LOW, 16)], [(SAME, 16)], [(RAW, 16)], [(RAW, 0), (LOW, 0), (SAME, 0), (LOW, 48)],  # the smallest, empty ones, an odd number of chunks
    [(LOW, 8192 - 16), (LOW, 8192), (LOW, 8192 + 16)],         # a workgroup's worth at one unit a lane, and either side of it
    [(SAME, 16384 - 16), (SAME, 16384), (SAME, 16384 + 16), (RAW, 4096), (RAW, 4112)],
    [(LOW, (640 << 10) + 16), (RAW, 48), (SAME, 1 << 20)],     # two units a lane
    [(LOW, 16384 - 16), (LOW, 16384 + 16), (RAW, 320 << 10)],
    [((RAW, LOW, SAME)[k % 3], 16 * (1 + 37 * k)) for k in range(64)],  # as many as a launch takes
])
@pytest.mark.parametrize("rows", [False, True])
def test_feed_pieces(spec, rows):
    gen = torch.Generator().manual_seed(len(spec) + 1000 * spec[0][1])
    pieces, dsts, wants, keep = _pieces(spec, gen)
    strided = (bz.FeedRows * 2)()
    src = torch.randint(256, (2, 9 * 26), generator=gen, dtype=torch.uint8).pin_memory()
    dst = torch.full((2, 9 * 890), 9, dtype=torch.uint8, device="cuda")
    for i in range(2):
        strided[i] = bz.FeedRows(src[i].data_ptr(), dst[i].data_ptr(), 9, 26, 26, 890)
    bz.check(bz.lib().bz_feed_pieces(pieces, len(spec), strided, 2 if rows else 0, bz._stream_ptr()))
    for got, want, piece in zip(dsts, wants, spec):
        assert torch.equal(got.cpu(), want), piece
    want = torch.full((2, 9, 890), 9, dtype=torch.uint8)
    if rows:
        want[:, :, :26] = src.view(2, 9, 26)
    assert torch.equal(dst.cpu().view(2, 9, 890), want)


def test_feed_pieces_refuses():
    buf = torch.zeros(64, dtype=torch.uint8).pin_memory()
    p, call = buf.data_ptr(), bz.lib().bz_feed_pieces
    many = (bz.FeedPiece * 65)()
    assert call(many, 65, None, 0, None) == bz.EINVAL
    for bad in ((p, p, 24, RAW), (p + 4, p, 16, LOW), (p, p + 8, 16, LOW), (None, p, 16, RAW), (None, p, 16, LOW), (p, None, 16, SAME), (p, p, 16, 3),
                (p, p, -16, SAME)):
        many[0] = bz.FeedPiece(*bad, 0)
        assert call(many, 1, None, 0, None) == bz.EINVAL, bad
