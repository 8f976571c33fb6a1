"""NN-Descent oracle (TEST INFRASTRUCTURE, never the product).

NN-Descent iterations in plain numpy: sampling, reverse lists, local join and
list update as nndescent.hip defines them (gpuknn/nndescent.cu:44-98, 293-346,
405-510, 1030-1326, 969-1028), one point after the other, on a matrix of squared
distances.  The order of everything is fixed, so the GPU's lists must be these.

Only tests/ may import this module.
"""
from __future__ import annotations

import numpy as np

from . import oracle as O

K = 32
INF = 0x7F800000
NONE = np.uint64(2**64 - 1)


def _rotation(key: int, it: int) -> int:
    return O.xorshift64star((key << 6) ^ ((it + 1) * 0x9E3779B97F4A7C15 & (2**64 - 1)))


def _key(bits, i) -> int:
    return int(bits) << 32 | int(i)


def init_random(B) -> list:
    """Lists of (key, is_new): 32 draws per point, repeats included.  B: the
    bits of the squared distances."""
    n = len(B)
    out = []
    for p in range(n):
        ids = [O.xorshift64star(p * K + j) % n for j in range(K)]
        ids = [(i + 1) % n if i == p else i for i in ids]
        out.append([(k, True) for k in sorted(_key(B[p, i], i) for i in ids)])
    return out


def init_merge(B, g1, g2) -> list:
    """knnmerge's start (gpuknn/knnmerge.cu:80-185): the first 16 ids of the own
    graph (old) and 16 draws from the other half (new)."""
    n1, n2 = len(g1), len(g2)
    out = []
    for p in range(n1 + n2):
        first = p < n1
        local = p if first else p - n1
        old = [int(i) if first else int(i) + n1 for i in (g1 if first else g2)[local][:K // 2]]
        draws = [O.xorshift64star(local * (K // 2) + t) for t in range(K // 2)]
        new = [r % n2 + n1 if first else r % n1 for r in draws]
        out.append(sorted([(_key(B[p, i], i), False) for i in old] + [(_key(B[p, i], i), True) for i in new]))
    return out


def _samples(lists, S, it, split):
    """Forward samples of every point: (new ids, old ids), S consecutive of a
    kind from a rotated rank where there are more."""
    out = []
    for p, row in enumerate(lists):
        ids = [(k & 0xFFFFFFFF, new) for k, new in row]
        new = [i for i, f in ids if f]
        old = [i for i, f in ids if not f and (split is None or (i < split) == (p < split))]
        h = _rotation(p, it)
        pick = []
        for kind, r in ((new, h & 0xFFFFFFFF), (old, h >> 32)):
            rot = r % len(kind) if len(kind) > S else 0
            pick.append([kind[(rot + j) % len(kind)] for j in range(min(S, len(kind)))])
        out.append(pick)
    return out


def descend(D, lists, S, keep, iterations, split=None, by_slot=False) -> list:
    """`iterations` of NN-Descent on the float32 squared distances D.  split: the
    merge form (old samples from the own half, new candidates take old partners
    only).  by_slot: equal distances go to the earlier candidate (new ones
    first, ascending ids) instead of the smaller id."""
    B = np.ascontiguousarray(D, np.float32).view(np.uint32).astype(np.uint64)
    n = len(D)
    for it in range(iterations):
        fwd = _samples(lists, S, it, split)
        rev = [([], []) for _ in range(n)]
        for p in range(n):
            for kind in (0, 1):
                for q in fwd[p][kind]:
                    rev[q][kind].append(p)
        bound = [np.float32(np.inf) if len(row) < K else np.uint32(row[K - 1][0] >> 32).view(np.float32)
                 for row in lists]
        props = [set() for _ in range(n)]
        for p in range(n):
            cand = []
            for kind in (0, 1):
                r = rev[p][kind]
                if len(r) > S:
                    rot = (_rotation(2 * p + kind, it) & 0xFFFFFFFF) % len(r)
                    r = [r[(j * len(r) // S + rot) % len(r)] for j in range(S)]
                cand.append(set(fwd[p][kind]) | set(r))
            new, old = sorted(cand[0] - cand[1]), sorted(cand[1])
            ids = np.array(new + old, np.int64)
            nn, nc = len(new), len(ids)
            if nc == 0:
                continue
            keys = (B[np.ix_(ids, ids)] << np.uint64(32)) | (np.arange(nc) if by_slot else ids).astype(np.uint64)
            is_new = np.arange(nc) < nn
            to_new = is_new[None, :] & ((split is None) | ~is_new[:, None]) & ~np.eye(nc, dtype=bool)
            to_old = is_new[:, None] & ~is_new[None, :]
            # (partners allowed, how many of the nearest are proposed)
            rounds = [(to_new, 1), (to_old, 1)] if keep == 0 else [(to_new | to_old, keep)]
            for allowed, most in rounds:
                near = np.argsort(np.where(allowed, keys, NONE), axis=1)[:, :most]
                for c in range(nc):
                    for j in near[c]:
                        if allowed[c, j] and D[ids[c], ids[j]] < bound[ids[c]]:
                            props[ids[c]].add(_key(B[ids[c], ids[j]], ids[j]))
        for t in range(n):
            have = {k for k, _ in lists[t]}
            lists[t] = [(k, k not in have) for k in sorted(have | props[t])[:K]]
    return lists


def arrays(lists):
    """(ids, distance bits) of the lists, n x 32; -1 and infinity's where a list is short."""
    ids = np.full((len(lists), K), -1, np.int64)
    bits = np.full((len(lists), K), INF, np.uint32)
    for p, row in enumerate(lists):
        ids[p, :len(row)] = [k & 0xFFFFFFFF for k, _ in row]
        bits[p, :len(row)] = [k >> 32 for k, _ in row]
    return ids, bits
