"""CPU enumeration of the sub-tile sweeps' mail records and of the store
wave's output (the address arithmetic of k_sweep_sub, restated): every face
value read is in range and is the record entry of the upstream cell beside the
pencil, written at an earlier step of its unit; every record entry read has one
writer; the two passes' resets cover every record; and the store wave writes
every slot of the box once, from the plane cell that holds that slot's value,
before the plane is reused."""
import itertools

import numpy as np
import pytest

KT, KS, KNB, KMAIL, KTHREADS, KPLANES = 16, 8, 4, 16, 256, 8


def batches(Bz):
    """Of a unit: its pencils' cells lie on Bz + 14 of the tile's steps."""
    return (Bz + 2 * (KS - 1) + KNB - 1) // KNB


def mail_of(ua, ub, nua, Bz):
    return (ub * nua + ua) * batches(Bz) * KNB * KMAIL


EXTENTS = [(1, 1, 1), (8, 9, 3), (17, 7, 2), (16, 41, 7), (32, 25, 9), (40, 31, 16), (24, 33, 33)]


def units(ex, ey, bwd):
    """The units that hold cells of an ex x ey box: (ua, ub) with the unit (A, B)
    of the sweep's frame, counted from its start corner over whole tiles."""
    nua, nub = -(-ex // KS), -(-ey // KS)
    na, nb_ = -(-ex // KT), -(-ey // KT)
    a0, b0 = (2 * na - nua, 2 * nb_ - nub) if bwd else (0, 0)
    return na, nb_, nua, nub, [(ua, ub, a0 + ua, b0 + ub)
                               for ua, ub in itertools.product(range(nua), range(nub))]


@pytest.mark.parametrize("bwd", [False, True])
@pytest.mark.parametrize("ex,ey,Bz", EXTENTS)
def test_mail_records(ex, ey, Bz, bwd):
    na, nb_, nua, nub, todo = units(ex, ey, bwd)
    size = mail_of(0, nub, nua, Bz)
    # what each entry holds: the cell (x, y, kk) in the sweep's frame, and its step
    entry = {}
    for ua, ub, A, B in todo:
        for lane in range(64):
            ui, uj = lane & 7, lane >> 3
            if ui != KS - 1 and uj != KS - 1:
                continue
            li, lj = KS * (A & 1) + ui, KS * (B & 1) + uj
            for w in range(batches(Bz) * KNB):
                e = mail_of(ua, ub, nua, Bz) + (uj if ui == KS - 1 else KS + ui) + w * KMAIL
                assert 0 <= e < size and e not in entry
                entry[e] = (KT * (A >> 1) + li, KT * (B >> 1) + lj, w - ui - uj)
    reads = 0
    for ua, ub, A, B in todo:
        sa, sb = A & 1, B & 1
        for lane in range(64):
            xf, st, m = lane < KNB * KS, (lane // KS) % KNB, lane % KS
            li, lj = (KS * sa, KS * sb + m) if xf else (KS * sa + m, KS * sb)
            up = ua > 0 if xf else ub > 0
            for n in range(batches(Bz)):
                w = n * KNB + st
                if not (up and w >= m and w - m < Bz):
                    continue
                e = mail_of(ua - 1, ub, nua, Bz) if xf else mail_of(ua, ub - 1, nua, Bz)
                e += (KS - 1 + w) * KMAIL + (m if (xf or m == KS - 1) else KS + m)
                x, y, kk = KT * (A >> 1) + li, KT * (B >> 1) + lj, w - m
                assert entry[e] == ((x - 1, y, kk) if xf else (x, y - 1, kk))
                reads += 1
    # every face between two units, once per cell of its pencils
    assert reads == ((nua - 1) * nub + (nub - 1) * nua) * KS * Bz


@pytest.mark.parametrize("word", [4, 8])
@pytest.mark.parametrize("bwd", [False, True])
@pytest.mark.parametrize("ex,ey,Bz", EXTENTS[:5])
def test_resets_and_output(ex, ey, Bz, bwd, word):
    nsteps = Bz + 2 * (KT - 1)
    na, nb_, nua, nub, todo = units(ex, ey, bwd)
    nbat = batches(Bz)
    reset = np.zeros(mail_of(0, nub, nua, Bz) * word, dtype=int)
    out = np.zeros(na * nb_ * nsteps * KTHREADS, dtype=int)
    dots = []
    vec = 16 // word
    per = 64 // vec
    for ua, ub, A, B in todo:
        sa, sb = A & 1, B & 1
        a, b = (na - 1 - (A >> 1), nb_ - 1 - (B >> 1)) if bwd else (A >> 1, B >> 1)
        psa, psb = (1 - sa, 1 - sb) if bwd else (sa, sb)
        w0 = KS * (sa + sb)
        tile0 = (b * na + a) * nsteps * KTHREADS
        dots.append((2 * b + psb) * nua + 2 * a + psa)
        for n in range(nbat):
            words = KNB * KMAIL * word // 16
            for lane in range(words):
                w = n * KNB + lane // (words // KNB)
                at = (mail_of(ua, ub, nua, Bz) + w * KMAIL) * word
                at += lane % (words // KNB) * 16
                reset[at:at + 16] += 1
            for j, lane in itertools.product(range(KNB * per // 64), range(64)):
                w, p = n * KNB + j * (64 // per) + lane // per, lane % per * vec
                if w >= nsteps - w0:
                    continue
                wp = nsteps - 1 - (w0 + w) if bwd else w0 + w
                slot = tile0 + wp * KTHREADS + (KS * psb + (p >> 3)) * KT + KS * psa + (p & 7)
                assert slot * word % 16 == 0
                for k in range(vec):
                    out[slot + k] += 1
                    # the slot's pencil, in the sweep's frame, is the plane cell's
                    lip, ljp = (slot + k) % KTHREADS % KT, (slot + k) % KTHREADS // KT
                    li, lj = (KT - 1 - lip, KT - 1 - ljp) if bwd else (lip, ljp)
                    ln = 63 - (p + k) if bwd else p + k
                    assert (li, lj) == (KS * sa + (ln & 7), KS * sb + (ln >> 3))
                # stored during batch n + 1; the plane is next written by step w + 8,
                # and its halos (read by step w + 9) one batch before that step's
                assert (w + KPLANES) // KNB > n + 1 and (w + KPLANES + 1) // KNB - 1 >= n + 1
    assert (reset == 1).all()
    # every cell of the units' pencils is stored once, no slot twice, and what
    # is stored besides is padding; one partial per unit
    slot = np.arange(out.size)
    lane, step, tile = slot % KTHREADS, slot // KTHREADS % nsteps, slot // KTHREADS // nsteps
    x, y = tile % na * KT + lane % KT, tile // na * KT + lane // KT
    kk = step - lane % KT - lane // KT
    inside = (x < nua * KS) & (y < nub * KS)
    assert (out[inside & (kk >= 0) & (kk < Bz)] == 1).all()
    assert (out[~inside] == 0).all() and out.max() == 1
    assert sorted(dots) == list(range(nua * nub))
