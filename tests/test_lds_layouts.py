"""Host-side check of the padded LDS row layouts of the asynchronous copies:

* stage_rows with an LDS row stride above the row bytes (chimere_amd/csrc/
  common.h), as the GEMV tile uses it (chimere_amd/csrc/tile_gemv.h,
  mmvq.hip: Q4_0 / Q8_0 / IQ3_S chunks, row padding 48 / 48 / 80 bytes);
* stage_row_spans with the tile's row stride for unaligned rows;
* the prefill GEMMs' stages (chimere_amd/csrc/prefill_gemm.h) and the slots of
  the plan's tile list (prefill.hip).

The slot -> (row, column) arithmetic is transcribed from the kernels.  Every
16-byte piece of every row must be written exactly once, no write may leave
its LDS buffer, no padding slot may be written, and the readers' furthest
byte (last block of the last row, plus the 4 bytes an unaligned 32-bit LDS
read may touch) must stay inside the buffer."""
import pytest

QK = 32
BYTES = {"q4_0": 18, "q8_0": 34, "iq3s": 110, "q6k": 210, "mxfp4": 17}
ELEMS = {"q4_0": 32, "q8_0": 32, "iq3s": 256, "q6k": 256, "mxfp4": 32}


def chunk_bytes(t, blocks):
    return blocks * QK // ELEMS[t] * BYTES[t]


def stage_rows_padded(nrows, seg, lseg, gstride, nthreads):
    """(lds byte offset, global byte offset) of every piece the padded path copies."""
    per, lper = seg // 16, lseg // 16
    tot = lper * nrows
    out = []
    for wave in range(nthreads // 64):
        for c0 in range(wave * 64, tot, (nthreads // 64) * 64):
            for lane in range(64):
                c = c0 + lane
                r, col = divmod(c, lper)
                if c < tot and col < per:
                    out.append((c0 * 16 + lane * 16, r * gstride + col * 16, r, col))
    return out


@pytest.mark.parametrize("t,pad", [("q4_0", 48), ("q8_0", 48), ("iq3s", 80)])
@pytest.mark.parametrize("ncols", [2048, 4096, 2048 + 512, 256 * 3])
def test_gemv_tile_padded_rows(t, pad, ncols):
    TILE_ROWS, CBLK, NTH = 16, 64, 256
    CB = chunk_bytes(t, CBLK)
    buf = TILE_ROWS * (CB + pad) + 16
    rb = ncols // ELEMS[t] * BYTES[t]
    nb = ncols // QK
    for b0 in range(0, nb, CBLK):
        cb = min(CBLK, nb - b0)
        seg = chunk_bytes(t, cb)
        goff = b0 * QK // ELEMS[t] * BYTES[t]
        padded = (seg | goff) % 16 == 0 and rb % 16 == 0
        if not padded:
            continue
        lseg = seg + pad
        for nr in (TILE_ROWS, 5, 1):
            pieces = stage_rows_padded(nr, seg, lseg, rb, NTH)
            seen = set()
            for lds, glob, r, col in pieces:
                assert 0 <= lds and lds + 16 <= buf
                assert lds == r * lseg + col * 16          # row r at r * lseg
                assert goff + glob + 16 <= nr * rb         # inside the nr rows of the matrix
                assert (r, col) not in seen
                seen.add((r, col))
            assert len(seen) == nr * (seg // 16)
            # furthest read: last byte of the last row's chunk + 4
            assert (nr - 1) * lseg + seg + 4 <= buf


# ---- prefill_gemm.h: the work-group's LDS and the copies into it

# blocks and bytes of a chunk
PF = {"q4_0": (8, 144), "q8_0": (4, 136), "iq3s": (8, 110), "q4k": (8, 144), "q5k": (8, 176), "q6k": (8, 210)}
EXPERT, SHARED, KQ = ("q4_0", "q8_0", "iq3s"), tuple(PF), ("q4k", "q5k")
PF_ROWS = 128


def pf_sl(t):
    return (PF[t][1] + 14 + 15) // 16 + (t in ("iq3s", "q6k", "q5k"))


def pf_skew(t):
    return pf_sl(t) % 2 == 0


def pf_row(t, r):
    return (r * pf_sl(t) + (r >> 2 if pf_skew(t) else 0)) * 16


def pf_wst(t):
    return pf_row(t, PF_ROWS) + 16


def pf_furthest(t, s):
    """End of the furthest LDS read of a row whose chunk starts at s (three whole
    words from the word that holds a field's first byte, two for a 32-bit one)."""
    w3, w2 = (lambda a: (a & ~3) + 12), (lambda a: (a & ~3) + 8)
    return max({"q4_0": lambda: [w3(s + 2 + 8 + 18 * 7), w3(s + 2 + 8 + 18 * 6)],
                "q8_0": lambda: [w3(s + 2 + 24 + 34 * 3), w3(s + 2 + 24 + 34 * 2)],
                "iq3s": lambda: [w2(s + 106), w2(s + 70), s + 74 + 4 * 7 + 4],
                "q4k": lambda: [w3(s + 16 + 24) + 96, w2(s + 12)],
                "q5k": lambda: [w3(s + 48 + 24) + 96, w2(s + 20 + 24)],
                "q6k": lambda: [w2(s + 128 + 32 + 24 + 4), s + 210]}[t]())


def pf_weight_pieces(t):
    """(instruction, lane) -> (row, column) of one chunk's copies, and each wave's
    number of instructions."""
    sl = pf_sl(t)
    nwg = (pf_row(t, PF_ROWS) // 16 + 63) // 64
    out = {}
    for g in range(nwg):
        for lane in range(64):
            cc = g * 64 + lane
            if pf_skew(t):
                g4, rem = divmod(cc, 4 * sl + 1)
                r, col = 4 * g4 + rem // sl, (rem % sl if rem < 4 * sl else sl)
            else:
                r, col = divmod(cc, sl)
            out[g, lane] = (r, col) if r < PF_ROWS and col < sl else None
    nwi = [(nwg - wave + 3) // 4 for wave in range(4)]
    assert nwi == [len([g for g in range(nwg) if g % 4 == w]) for w in range(4)]
    return nwg, out


@pytest.mark.parametrize("t", SHARED)
def test_prefill_weight_stage(t):
    """Rows whose chunks start at any even place of a 16-byte granule: every piece
    of every row's span is copied once to its row's slots, inside the stage; every
    copy instruction of a wave has an active lane (the waits count them); no read
    of a row leaves the stage or the bytes copied for it, but for the words'
    padding, which is inside the stage."""
    cb = PF[t][1]
    nwg, pieces = pf_weight_pieces(t)
    for phase, stride in [(p, s) for p in range(0, 16, 2) for s in (0, 2, 14)]:
        seen, active = set(), {g: 0 for g in range(nwg)}
        for (g, lane), rc in pieces.items():
            if rc is None:
                continue
            r, col = rc
            pre = (phase + r * stride) % 16
            if col * 16 < pre + cb:
                active[g] += 1
                dst = g * 1024 + lane * 16
                assert dst == pf_row(t, r) + 16 * col and dst + 16 <= pf_wst(t) - 16
                assert (r, col) not in seen
                seen.add((r, col))
        assert all(active.values())
        assert seen == {(r, c) for r in range(PF_ROWS) for c in range(((phase + r * stride) % 16 + cb + 15) // 16)}
        for r in range(PF_ROWS):
            s = pf_row(t, r) + (phase + r * stride) % 16
            assert s + cb <= pf_row(t, r) + 16 * pf_sl(t)
            assert pf_furthest(t, s) <= pf_wst(t)


def pf_work_group(launch, te, ts, mt):
    """(stages, bytes of a weight stage, 16-pair x block units of an activation
    stage) of a kernel's LDS, and its runs: (type, pair tiles, activation blocks
    per stage, two weight stages)."""
    one = mt == 2 and not (launch == "down" and ts in KQ + ("q6k",))
    wide = pf_wst(ts) > pf_wst(te) and (one or (pf_sl(ts) <= 10 and ts not in KQ))
    wst2 = pf_wst(ts if wide else te)
    xu = 16 if mt == 2 and not one else 4 * mt
    runs = []
    for t in {te, ts}:
        most = 2 if t == "q6k" else (4 if launch == "gate_up" else 2) if t in KQ else 4
        m = min(mt, most)
        for k in {m} if m < mt else {mt, max(1, mt // 2)}:
            runs.append((t, k, 8 if PF[t][0] == 8 and k == 2 and not one else 4, not one and pf_wst(t) <= wst2))
    return 1 if one else 2, wst2, xu, runs


@pytest.mark.parametrize("launch", ["gate_up", "down"])
@pytest.mark.parametrize("mt", [1, 2, 4])
def test_prefill_work_group_lds(launch, mt):
    """Every type x tile size run by a kernel fits its LDS: the weight stages, the
    activation and scale stages, the wave's copies of the row list (in the second
    activation stage) and the epilogue's exchange (in the scale stages)."""
    for te, ts in [(te, ts) for te in EXPERT for ts in SHARED]:
        nw, wst2, xu, runs = pf_work_group(launch, te, ts, mt)
        sd = (4 if ts in KQ else 2) * xu * 16                      # words
        total = nw * wst2 + 2 * xu * 1024 + 4 * sd + (4096 if "iq3s" in (te, ts) else 16)
        assert total <= 160 * 1024 // (3 if mt == 2 and nw == 1 else 2)
        for t, m, xb, wdb in runs:
            assert 2 * pf_wst(t) <= nw * wst2 if wdb else pf_wst(t) <= nw * wst2
            assert PF[t][0] % xb == 0 and m * xb <= xu
            assert 16 * m * xb <= xu * 16
            assert 4 * 64 * 4 <= xu * 1024 and 16 * m <= 64        # the list holds 64 rows
            assert 4 * 16 * m <= sd


@pytest.mark.parametrize("mt,xb", [(1, 4), (2, 4), (2, 8), (4, 4)])
def test_prefill_activation_stage(mt, xb):
    """The pieces that the copies leave in an activation stage, and the words in a
    scale stage, are those the lanes read: each piece copied once."""
    nxp, nxb = (mt // 2, xb // 2) if mt > 1 else (1, xb // 4)
    lds, sc = {}, {}
    for wave in range(4):
        for lane in range(64):
            for j in range(nxp):
                grp, r = (wave + 4 * j if mt > 1 else wave & 1), lane >> 3
                for k in range(nxb):
                    unit = xb // 2 * (wave + 4 * j) + k if mt > 1 else xb // 2 * (wave & 1) + nxb * (wave >> 1) + k
                    off = (0 if mt > 1 else 128 * nxb * (wave >> 1)) + 16 * ((lane & 7) ^ r) + 128 * k
                    at = unit * 1024 + lane * 16
                    assert at not in lds and at + 16 <= mt * xb * 1024
                    lds[at] = (8 * grp + r, off)              # pair, byte of its row's stage
    assert sorted(lds.values()) == [(p, o) for p in range(16 * mt) for o in range(0, 64 * xb, 16)]
    for lane in range(16 * mt):
        for k in range(xb // 4):
            for i in range(4):
                sc[64 * mt * k + 4 * lane + i] = (lane, 4 * k + i)
    assert sorted(sc) == list(range(16 * mt * xb))
    kt = 4 // mt
    for q in range(4):
        for c in range(16):
            xo = (c >> 3) * (512 * xb) + (c & 7) * 128 + (q ^ (c & 7)) * 16
            for b in range(xb):
                for m in range(mt):
                    at = m * (1024 * xb) + (b >> 1) * 1024 + (xo ^ 64 if b & 1 else xo)
                    assert lds[at] == (16 * m + c, 64 * b + 16 * q)
                    for i in range(4):
                        assert sc[(16 * m + 4 * q + i) * 4 + 64 * mt * (b >> 2) + (b & 3)] == (16 * m + 4 * q + i, b)
                if b % kt == 0:
                    assert sc[64 * mt * (b >> 2) + (b & 3) + (16 * (q % mt) + c) * 4 + q // mt] == \
                        (16 * (q % mt) + c, b + q // mt)


def eighth(n):
    return (n + 7) >> 3


def pf_place(block, nslice, nsh, ne, whole):
    """(tile, slice) of a work-group, shared tiles before the experts'; None: no work."""
    x, k = block & 7, block >> 3
    if whole:
        g, sl = divmod(k, nslice)
        per, persh = max(eighth(ne), 1), eighth(nsh)
        slots = {s: s for s in range(nsh)}
        slots.update({8 * (persh + t - t // per * per) + t // per: nsh + t for t in range(ne)})
        t = slots.get(8 * g + x)
        return None if t is None else (t, sl)
    ps = eighth(nsh * nslice)
    n, i = (nsh * nslice, k) if k < ps else (ne * nslice, k - ps)
    w = x * eighth(n) + i
    return None if i >= eighth(n) or w >= n else (w // nslice + (0 if k < ps else nsh), w % nslice)


@pytest.mark.parametrize("tp", [16, 32, 64])
@pytest.mark.parametrize("E,K,T", [(1, 1, 1), (4, 2, 33), (8, 8, 130), (64, 4, 12), (256, 8, 9), (300, 12, 70),
                                   (1024, 16, 65)])
def test_prefill_tile_dealing(tp, E, K, T):
    """However the router deals the pairs, the plan's tiles fit their list, every
    slice of every tile belongs to one work-group of the launch, and (but for
    whole tiles) no XCD has more than an eighth, rounded up, of either part's."""
    import random
    rng = random.Random(E * K + T)
    tiles = lambda n: T * K // n + min(T * K, E)  # noqa: E731
    entries = tiles(16) + (T + 15) // 16 + 16                   # of the workspace
    for shared, nslice in ((False, 4), (True, 16), (True, 1), (True, 3)):
        for case in range(3):
            counts = [0] * E
            for _ in range(T):
                for e in (range(K) if case == 0 else rng.sample(range(E), K)):
                    counts[e] += 1
            if case == 1:                                       # one pair left over everywhere it can be
                counts = [tp + 1 if i < T * K // (tp + 1) else 0 for i in range(E)]
            ne = sum((c + tp - 1) // tp for c in counts)
            nsh = (T + tp - 1) // tp if shared else 0
            assert ne <= tiles(tp)
            assert 1 + nsh + ne <= entries and 8 * (eighth(nsh) + eighth(tiles(tp))) <= entries
            want = sorted((t, s) for t in range(nsh + ne) for s in range(nslice))
            for whole in (False, True):
                grid = (8 * (eighth(nsh) + eighth(tiles(tp))) * nslice if whole else
                        8 * (eighth(nsh * nslice) + eighth(tiles(tp) * nslice)))
                if grid > 20000:
                    continue
                got = [(b & 7, pf_place(b, nslice, nsh, ne, whole)) for b in range(grid)]
                assert sorted(p for _, p in got if p) == want
                if not whole:
                    for part in (lambda t: t < nsh, lambda t: t >= nsh):
                        load = [sum(1 for x, p in got if p and x == k and part(p[0])) for k in range(8)]
                        assert max(load) == eighth(sum(load)) and load == sorted(load, reverse=True)


@pytest.mark.parametrize("t", ["iq3s", "q6k", "mxfp4"])
def test_gemv_row_spans(t):
    """stage_row_spans (common.h) into the GEMV tile (mmvq_tile, mmvq.hip): whole
    and ragged chunks, rows at any place of a granule (MXFP4: odd ones too)."""
    pad = {"iq3s": 80}.get(t, 0)
    cb = chunk_bytes(t, 64)
    tile = 16 * (cb + max(pad, ((cb + 30) & ~15) - cb)) + 16
    for blocks in {"mxfp4": range(1, 65, 7)}.get(t, range(8, 65, 8)):
        seg = chunk_bytes(t, blocks)
        ss = (seg + 30) & ~15
        per = ss >> 4
        for rb in {seg, 3 * seg, seg + 7 * BYTES[t]}:
            for phase in range(0, 16, 1 if t == "mxfp4" else 2):
                for nr in (16, 5, 1):
                    seen = {}
                    for c in range(per * nr):
                        r, col = divmod(c, per)
                        pre = (phase + r * rb) % 16
                        if col * 16 < pre + seg:
                            assert c * 16 + 16 <= tile - 16
                            seen[r] = seen.get(r, 0) + 1
                            assert c * 16 == r * ss + col * 16
                    assert seen == {r: ((phase + r * rb) % 16 + seg + 15) // 16 for r in range(nr)}
                    # a row's bytes in its LDS row, its last 32-bit read inside the tile
                    assert all((phase + r * rb) % 16 + seg <= ss for r in range(nr))
                    assert (nr - 1) * ss + (phase + (nr - 1) * rb) % 16 + seg + 7 <= tile


@pytest.mark.parametrize("pre", [0, 2, 4, 6, 8, 10, 12, 14])
def test_spans_in_288_byte_slots(pre):
    """stage_spans (common.h) with 18 LDS slots per row, as the double-buffered
    tile stages 16-block IQ3_S chunks (two 110-byte superblocks, starting
    `pre` bytes into a 16-byte granule): 64 rows fit the 18,448-byte buffer,
    every piece of every row once, reads of a row's chunk inside its slot."""
    seg, nrows, minper, TB = 220, 64, 18, 64 * 16 * 18 + 16
    per0 = (pre + seg + 15) >> 4
    per = max(per0, minper)
    assert nrows * per * 16 <= TB
    seen = set()
    for c in range(per * nrows):
        r, col = divmod(c, per)
        if col < per0:
            assert c * 16 == r * per * 16 + col * 16
            seen.add((r, col))
    assert len(seen) == nrows * per0
    # the chunk's last byte (plus a 4-byte unaligned read) stays in the row's slot
    assert pre + seg + 4 <= per * 16


def test_iq3s_sign_folded_codebook_lookup():
    """The one-token expert kernel's IQ3_S lookups in the sign-folded codebook
    (chimere_amd/csrc/common.h: Iq3sSignedGrid, iq3s_levels<true>): entry
    16 i + n is entry i with byte k negated where bit k of n is set, and the
    byte offsets (pr << 6) | ((s * 0x4004) & 0x3C003C) of a perm-packed index
    pair give entries 16 idx + nibble in both 16-bit halves.  Checked against
    the codebook with the signs applied per byte (the decode every other kernel
    and the oracle use), for every entry and sign nibble, and on random blocks."""
    import numpy as np
    import npref
    G = npref.GRID.astype(np.int64)
    tab = np.zeros(8192, np.int64)
    for n in range(16):
        v = np.zeros(512, np.int64)
        for k in range(4):
            b = (G >> (8 * k)) & 255
            v |= (np.where((n >> k) & 1, (256 - b) & 255, b)) << (8 * k)
        tab[np.arange(512) * 16 + n] = v
    for n in range(16):   # every entry, every sign nibble: signed levels
        for k in range(4):
            lv = (G >> (8 * k)) & 255
            got = ((tab[np.arange(512) * 16 + n] >> (8 * k)) & 255).astype(np.int8).astype(np.int64)
            assert (got == np.where((n >> k) & 1, -lv, lv)).all()

    def perm(src0, src1, sel):   # v_perm_b32 with selectors 0..7 (bytes of src1, then src0)
        b = [(src1 >> (8 * i)) & 255 for i in range(4)] + [(src0 >> (8 * i)) & 255 for i in range(4)]
        return sum(b[(sel >> (8 * i)) & 255] << (8 * i) for i in range(4))

    def nib_bits(n):
        return (n * 0x00204081) & 0x01010101

    rng = np.random.default_rng(5)
    for _ in range(2000):
        qs = [int(x) for x in rng.integers(0, 256, 8)]
        qh, sg = int(rng.integers(0, 256)), int(rng.integers(0, 1 << 32))
        qs0 = qs[0] | qs[1] << 8 | qs[2] << 16 | qs[3] << 24
        qs1 = qs[4] | qs[5] << 8 | qs[6] << 16 | qs[7] << 24
        h0, h1 = nib_bits(qh & 15), nib_bits((qh >> 4) & 15)
        for p in range(4):
            pr = perm(h0 if p < 2 else h1, qs0 if p < 2 else qs1, 0x07030602 if p & 1 else 0x05010400)
            t = (((sg >> (8 * p)) & 255) * 0x4004) & 0x003C003C
            ab = ((pr << 6) | t) & 0xFFFFFFFF
            for half, word in ((ab & 0xFFFF, 2 * p), (ab >> 16, 2 * p + 1)):
                assert half % 4 == 0 and half < 32768
                idx = qs[word] | ((qh >> word) & 1) << 8          # entry of word `word`
                nib = (sg >> (4 * word)) & 15                     # its sign nibble
                assert half // 4 == 16 * idx + nib
                want = 0
                for k in range(4):
                    lv = (int(G[idx]) >> (8 * k)) & 255
                    want |= (((256 - lv) & 255) if (nib >> k) & 1 else lv) << (8 * k)
                assert int(tab[half // 4]) == want
