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


def mail_of(A, B, nsa, nsteps):
    return (B * nsa + A) * (-(-nsteps // KNB) * KNB) * KMAIL  # whole batches


@pytest.mark.parametrize("na,nb_,Bz", [(1, 1, 1), (1, 1, 3), (2, 1, 2), (1, 3, 7), (2, 2, 9),
                                       (3, 2, 16), (2, 3, 33)])
def test_mail_records(na, nb_, Bz):
    nsa, nsb, nsteps = 2 * na, 2 * nb_, Bz + 2 * (KT - 1)
    size = mail_of(0, nsb, nsa, nsteps)
    # what each entry holds: the cell (x, y, kk) in the sweep's frame, and its step
    entry = {}
    for A, B in itertools.product(range(nsa), range(nsb)):
        for lane in range(64):
            ui, uj = lane & 7, lane >> 3
            if ui != KS - 1 and uj != KS - 1:
                continue
            li, lj = KS * (A & 1) + ui, KS * (B & 1) + uj
            for w in range(-(-nsteps // KNB) * KNB):
                e = mail_of(A, B, nsa, nsteps) + (uj if ui == KS - 1 else KS + ui) + w * KMAIL
                assert 0 <= e < size and e not in entry
                entry[e] = (KT * (A >> 1) + li, KT * (B >> 1) + lj, w - li - lj)
    reads = 0
    nbat = (nsteps + KNB - 1) // KNB
    for A, B in itertools.product(range(nsa), range(nsb)):
        sa, sb = A & 1, B & 1
        for lane in range(64):
            xf, st, m = lane < KNB * KS, (lane // KS) % KNB, lane % KS
            li, lj = (KS * sa, KS * sb + m) if xf else (KS * sa + m, KS * sb)
            up = A > 0 if xf else B > 0
            ahead = -1 if (sa if xf else sb) else KT - 1
            off = li + lj
            for n in range(nbat):
                w = n * KNB + st
                if not (up and w < nsteps and off <= w and w - off < Bz):
                    continue
                src = mail_of(A - 1, B, nsa, nsteps) if xf else mail_of(A, B - 1, nsa, nsteps)
                src += m if (xf or m == KS - 1) else KS + m
                e = src + (w + ahead) * KMAIL
                assert 0 <= w + ahead < nsteps
                x, y, kk = KT * (A >> 1) + li, KT * (B >> 1) + lj, w - off
                assert entry[e] == ((x - 1, y, kk) if xf else (x, y - 1, kk))
                reads += 1
    # every face between two units, once per cell of its pencils
    assert reads == ((nsa - 1) * nsb + (nsb - 1) * nsa) * KS * Bz


@pytest.mark.parametrize("word", [4, 8])
@pytest.mark.parametrize("bwd", [False, True])
@pytest.mark.parametrize("na,nb_,Bz", [(1, 1, 1), (2, 1, 2), (1, 2, 7), (2, 2, 9)])
def test_resets_and_output(na, nb_, Bz, bwd, word):
    nsa, nsb, nsteps = 2 * na, 2 * nb_, Bz + 2 * (KT - 1)
    nbat = (nsteps + KNB - 1) // KNB
    reset = np.zeros(mail_of(0, nsb, nsa, nsteps) * word, dtype=int)
    out = np.zeros(na * nb_ * nsteps * KTHREADS, dtype=int)
    vec = 16 // word
    per = 64 // vec
    for A, B in itertools.product(range(nsa), range(nsb)):
        sa, sb = A & 1, B & 1
        a, b = (na - 1 - (A >> 1), nb_ - 1 - (B >> 1)) if bwd else (A >> 1, B >> 1)
        psa, psb = (1 - sa, 1 - sb) if bwd else (sa, sb)
        tile0 = (b * na + a) * nsteps * KTHREADS
        for n in range(nbat):
            words = KNB * KMAIL * word // 16
            for lane in range(words):
                w = n * KNB + lane // (words // KNB)
                if w < nsteps:
                    at = (mail_of(A, B, nsa, nsteps) + w * KMAIL) * word
                    at += lane % (words // KNB) * 16
                    reset[at:at + 16] += 1
            for j, lane in itertools.product(range(KNB * per // 64), range(64)):
                w, p = n * KNB + j * (64 // per) + lane // per, lane % per * vec
                if w >= nsteps:
                    continue
                wp = nsteps - 1 - w if bwd else w
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
    per_unit = reset.reshape(nsa * nsb, -1)[:, :nsteps * KMAIL * word]
    assert (per_unit == 1).all() and reset.max() == 1 and (out == 1).all()
