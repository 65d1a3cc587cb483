"""Model of the SpMM kernels' chunk decode (flashx_amd/csrc/spmm.hip,
decode_chunk), run on the CPU against oracle-built images.  Each of 64 lanes
takes 8 words of a 512-word chunk.  A tile header is 8 words long and a tile at
least 11, so a lane's entries all belong to the last tile that starts at or
before its first item word: its words are described by two 8-bit masks
(row heads and entries).  The lane a tile starts in comes from the directory
window, one entry per lane; an entry's value position (weighted images) from
the number of entries decoded before its tile's first lane.  The stream must
equal a plain sequential decode, for whole block rows and for items cut at
arbitrary words (binary) or tile starts (weighted)."""
import numpy as np
import pytest

from test_decode_model import seq_decode, seq_decode_w, tiles_of, tiles_of_w

SENT = 0x7FFFFFFF


def clamp8(x):
    return max(0, min(8, x))


def mask_decode(words, bw, d, begin, pend, carry, log2w, vw=0):
    """Entries (row, column[, value word]) of item words [begin, pend) of the
    block row at word bw; d: (start, block column[, values word]) per tile."""
    out, c0, c = [], 0, (bw + begin) & ~7
    ct = max(i for i, e in enumerate(d) if e[0] <= begin)
    while c < bw + pend:
        cb = c - bw
        live = [ct + t < len(d) for t in range(64)]
        win = [d[ct + t] if live[t] else (SENT, 0, 0) for t in range(64)] + [(SENT, 0, 0)]
        first = [0 if t == 0 else (win[t][0] - cb + 7) >> 3 for t in range(64)]  # lane a tile begins with
        begins = [f for t, f in enumerate(first) if live[t] and f < 64]
        assert begins[0] == 0 and all(a < b for a, b in zip(begins, begins[1:]))
        M = sum(1 << f for f in begins)
        lanes, row_in = [], []
        for l in range(64):
            p0, below = cb + 8 * l, M & ((2 << l) - 1)
            j = bin(below).count("1") - 1
            lo = max(clamp8(begin - p0), clamp8(win[j][0] + 8 - p0))
            hi = min(clamp8(pend - p0), clamp8(win[j + 1][0] - p0))
            if vw:
                hi = min(hi, clamp8(win[j][2] - p0))
            body = ((1 << max(hi - lo, 0)) - 1) << lo
            ws = [int(words[c + 8 * l + i]) if c + 8 * l + i < len(words) else 0 for i in range(8)]
            h8 = sum((w >> 15) << i for i, w in enumerate(ws))
            heads = body & h8
            last = ws[heads.bit_length() - 1] & 0x7FFF if heads else -1
            lanes.append((ws, heads, body & ~h8, last, j, below.bit_length() - 1))
        for l in range(64):
            row_in.append(next((lanes[m][3] for m in range(l - 1, -1, -1) if lanes[m][1]), carry))
        carry = next((lanes[m][3] for m in range(63, -1, -1) if lanes[m][1]), carry)
        excl = np.concatenate([[0], np.cumsum([bin(e[2]).count("1") for e in lanes])]).astype(int)
        for l, (ws, heads, ents, _, j, fl) in enumerate(lanes):
            r, o = row_in[l], int(excl[l])
            for i in range(8):
                if heads >> i & 1:
                    r = ws[i] & 0x7FFF
                if ents >> i & 1:
                    e = (r, (win[j][1] << log2w) | ws[i])
                    qt = -c0 if j == 0 else int(excl[fl])
                    out.append(e + (win[j][2] + (o - qt) * vw,) if vw else e)
                    o += 1
        cn = c + 512
        adv = sum(1 for t in range(64) if live[t] and win[t][0] <= cn - bw)
        qn, fj = int(excl[64]), first[adv - 1]
        c0 = c0 + qn if adv == 1 else (0 if fj >= 64 else qn - int(excl[fj]))
        if cn < bw + pend:
            ct += adv - 1
        c = cn
    return out


@pytest.mark.parametrize("scale,lh,lw,ef", [(10, 5, 6, 16), (10, 7, 10, 4), (11, 4, 4, 16), (9, 9, 9, 16), (12, 6, 15, 16)])
def test_mask_decode(orc, scale, lh, lw, ef):
    rng = np.random.default_rng(scale * 100 + lh)
    s, dd = orc.rmat_edges(scale, ef << scale, scale)
    img = orc.build_2d(s, dd, n=1 << scale, log2h=lh, log2w=lw, flags=orc.DEDUP)
    words, offs = np.frombuffer(img.data, dtype=np.uint16), img.offs
    for br in range(0, len(offs) - 1, max(1, (len(offs) - 1) // 16)):
        bs, be = offs[br] // 2, offs[br + 1] // 2
        d = [tuple(int(x) for x in e) for e in tiles_of(words, bs, be)]
        cuts = sorted(set([0, be - bs] + [int(x) for x in rng.integers(0, be - bs, size=3)]))
        for a0, a1 in zip(cuts[:-1], cuts[1:]):
            _, carry = seq_decode(words[bs:be], d, 0, a0, -1, lw)
            ref, _ = seq_decode(words[bs:be], d, a0, a1, carry, lw)
            assert mask_decode(words, int(bs), d, int(a0), int(a1), int(carry), lw) == ref, (br, a0, a1)


@pytest.mark.parametrize("dt,lh,lw", [(np.float32, 5, 6), (np.float64, 7, 10), (np.int32, 4, 4), (np.int64, 6, 5)])
def test_mask_decode_weighted(orc, dt, lh, lw):
    rng = np.random.default_rng(lh * 7 + lw)
    s, dd = orc.rmat_edges(10, 16 << 10, lh)
    img = orc.build_2d_w(s, dd, (rng.random(len(s)) * 10).astype(dt), n=1 << 10, log2h=lh, log2w=lw, flags=orc.DEDUP)
    vw = np.dtype(dt).itemsize // 2
    words, offs = np.frombuffer(img.data, dtype=np.uint16), img.offs
    for br in range(0, len(offs) - 1, max(1, (len(offs) - 1) // 16)):
        bs, be = offs[br] // 2, offs[br + 1] // 2
        d = [tuple(int(x) for x in e) for e in tiles_of_w(words, bs, be, vw)]
        cuts = sorted(set([0, be - bs] + [d[int(x)][0] for x in rng.integers(0, len(d), size=3)]))
        for a0, a1 in zip(cuts[:-1], cuts[1:]):
            ref = seq_decode_w(words[bs:be], d, a0, a1, lw, vw)
            assert mask_decode(words, int(bs), d, int(a0), int(a1), -1, lw, vw) == ref, (br, a0, a1)
