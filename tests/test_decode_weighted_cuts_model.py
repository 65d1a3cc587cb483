"""Model of how the SpMM kernels walk a weighted image's items
(flashx_amd/csrc/spmm.hip, decode_chunk and fetch_next; the cuts of
fmx_core.cpp's get_plan and image_dev.hip's fix_items), run on the CPU
against oracle-built images.  An item may start inside a tile's entries: it
brings the row in force there and the number of the tile's entries before
it, from which the places of its values count.  The walk steps from inside a
tile's values straight to the next tile.  The items' entries, one item after
the other, must be the plain sequential decode's, each with its value word;
and no chunk that lies in values alone may be visited."""
import numpy as np
import pytest

from test_decode_masks_model import SENT, clamp8
from test_decode_model import tiles_of_w


def sequential(words, d, log2w, vw):
    """Entries of a block row as (word, tile, row, column, value word)."""
    out = []
    for t, (x, bc, v) in enumerate(d):
        row, n = -1, 0
        for p in range(x + 8, v):
            w = int(words[p])
            if w & 0x8000:
                row = w & 0x7FFF
            else:
                out.append((p, t, row, (bc << log2w) | w, v + n * vw))
                n += 1
    return out


def cut_at(d, words, p):
    """Where a cut at word p moves: to its share of the tile's entry words."""
    t = max(i for i, e in enumerate(d) if e[0] <= p)
    x, _, v = d[t]
    end = d[t + 1][0] if t + 1 < len(d) else words
    return t, x + 8 + (p - x) * (v - x - 8) // (end - x)


def start_of(words, d, t, p):
    """The row in force at word p of tile t (-1 at a header) and the tile's
    entries before it."""
    x, _, v = d[t]
    before = sum(1 for q in range(x + 8, p) if not words[q] & 0x8000)
    if p >= v or words[p] & 0x8000:
        return -1, before
    q = max(q for q in range(x + 8, p) if words[q] & 0x8000)
    return int(words[q]) & 0x7FFF, before


def walk(words, bw, d, t0, begin, pend, carry, before, log2w, vw):
    """Entries (row, column, value word) of item [begin, pend), and the chunks
    visited."""
    out, chunks, c0, ct = [], [], before, t0
    abs_end, c = bw + pend, (bw + begin) & ~7
    while c < abs_end:
        chunks.append(c - bw)
        cb = c - bw
        live = [ct + t < len(d) for t in range(64)]
        win = [d[ct + t] if live[t] else (SENT, 0, 0) for t in range(64)] + [(SENT, 0, 0)]
        first = [0 if t == 0 else (win[t][0] - cb + 7) >> 3 for t in range(64)]
        begins = {f for t, f in enumerate(first) if live[t] and f < 64}
        assert len(begins) == sum(1 for t, f in enumerate(first) if live[t] and f < 64) and 0 in begins
        qn, q0, j, row = 0, -c0, -1, carry
        for lane in range(64):
            if lane in begins:
                j += 1
                q0 = -c0 if j == 0 else qn
            p0 = cb + 8 * lane
            x, bc, v = win[j]
            lo = clamp8(max(x + 8, begin) - p0)
            hi = clamp8(min(win[j + 1][0], pend, v) - p0)
            for p in range(p0 + lo, p0 + hi):
                w = int(words[bw + p])
                if w & 0x8000:
                    row = w & 0x7FFF
                else:
                    out.append((row, (bc << log2w) | w, v + (qn - q0) * vw))
                    qn += 1
        carry, tiles, qt = row, j + 1, q0
        cn = c + 512
        if cn < abs_end:
            pn = cn - bw
            adv = sum(1 for t in range(64) if live[t] and win[t][0] <= pn)
            if adv < 64 and pn >= win[adv - 1][2]:
                to = (bw + win[adv][0]) & ~7 if live[adv] else abs_end
                if to > cn:
                    cn = min(to, abs_end)
                    if cn < abs_end:
                        adv = sum(1 for t in range(64) if live[t] and win[t][0] <= cn - bw)
            if cn < abs_end:
                c0 = 0 if adv > tiles else qn - qt
                ct += adv - 1
        c = cn
    return out, chunks


@pytest.mark.parametrize("dt,lh,lw,hub", [(np.float32, 5, 6, 0), (np.float64, 6, 10, 0), (np.int32, 4, 4, 0),
                                          (np.int64, 6, 10, 900), (np.float32, 10, 10, 1000), (np.float64, 3, 10, 1024)])
def test_items_cut_inside_tiles(orc, dt, lh, lw, hub):
    """hub: a row of that many entries, whose row part spans several chunks."""
    rng = np.random.default_rng(lh * 31 + lw)
    n = 1 << 10
    s, dd = orc.rmat_edges(10, 16 << 10, lh)
    s = np.concatenate([s, np.full(hub, 5, s.dtype)])
    dd = np.concatenate([dd, np.arange(hub).astype(dd.dtype)])
    img = orc.build_2d_w(s, dd, (rng.random(len(s)) * 10).astype(dt), n=n, log2h=lh, log2w=lw, flags=orc.DEDUP)
    vw = np.dtype(dt).itemsize // 2
    words, offs = np.frombuffer(img.data, dtype=np.uint16).astype(np.int64), img.offs
    inside = skipped = 0
    for br in range(0, len(offs) - 1, max(1, (len(offs) - 1) // 12)):
        bs, be = int(offs[br] // 2), int(offs[br + 1] // 2)
        d = [tuple(int(x) for x in e) for e in tiles_of_w(words, bs, be, vw)]
        ref = sequential(words[bs:be], d, lw, vw)
        for pieces in (1, 2, 5, max(1, (be - bs) // 40)):
            ends = [cut_at(d, be - bs, (be - bs) * i // pieces) for i in range(1, pieces)]
            ends = [(0, 0)] + ends + [(len(d), be - bs)]
            assert all(a[1] <= b[1] for a, b in zip(ends[:-1], ends[1:]))
            got = []
            for (t, a), (_, b) in zip(ends[:-1], ends[1:]):
                if a == b:
                    continue
                carry, before = start_of(words[bs:be], d, t, a) if a else (-1, 0)
                inside += carry >= 0
                entries, chunks = walk(words, bs, d, t, a, b, carry, before, lw, vw)
                got += entries
                for c in chunks[1:]:  # no chunk starts in values that reach past its end
                    u = max(i for i, e in enumerate(d) if e[0] <= max(c, 0))
                    nxt = d[u + 1][0] if u + 1 < len(d) else be - bs
                    assert c < d[u][2] or nxt < c + 512
                skipped += len(range(chunks[0], b, 512)) > len(chunks)
            same = got == [e[2:] for e in ref]  # (no list in the assertion: its diff takes minutes)
            assert same, (br, pieces)
    assert inside > 0 and (skipped > 0 or not hub)
