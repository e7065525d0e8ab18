"""CPU emulation of the PCG's reduction from items (cloth_sim_self_collision_amd/
csrc/cs_item_sum.hpp: tile_items, add_items, chain_items, walk_tile), step for
step, recording every index the kernel reads or writes.  As for the reduction
with one summary per tile (test_sum_emulation.py) it checks that every index
stays inside its buffer and that the emulated result is the left-to-right loop
of the reference's InnerProduct (matrix_square_sparse.cpp:313-325) bit for bit.
Integer arithmetic wraps at 64 bits as on the device."""
import math

import numpy as np
import pytest

from test_sum_emulation import (K_SUM_BLOCK, K_SUM_BUF, K_SUM_PER, K_SUM_TILE, Bounds, _cases,
                                _sequential, sign_exp, sum_normal, sum_tiles, wave_walk, wrap64)

# constants of cs_item_sum.hpp
K_ITEM_CAP = 256
K_ITEM_WIN = 512
K_ITEM_PASS = 4
K_ITEM_NONE = -2
HUGE = 1 << 60
LL_MAX, LL_MIN = (1 << 63) - 1, -(1 << 63)


def normal_code(s):
    return sign_exp(s) if sum_normal(s) else -1


def code_exp(code):
    return (code & 0x7ff) - 1023


def _ldexp(x, e):
    with np.errstate(all="ignore"):
        return float(np.ldexp(np.float64(x), e))


def tile_items(t, n, b, approx, bnd):
    """The items of tile b, or None when they are more than K_ITEM_CAP."""
    e0 = b * K_SUM_TILE
    real = min(n - e0, K_SUM_TILE) if n > e0 else 0
    if real:
        bnd.see("t", np.arange(e0, e0 + real))
    x = np.zeros(K_SUM_TILE)
    x[:real] = t[e0:e0 + real]
    with np.errstate(all="ignore"):
        # a thread's prediction before its first addend is formed apart from
        # the one after its neighbour's last: as incl - run on the device
        per = x.reshape(K_SUM_BLOCK, K_SUM_PER)
        loc = np.cumsum(per, axis=1)
        incl = np.cumsum(loc[:, -1])
        base = approx + (incl - loc[:, -1])
    q, single, cb, ca = [0] * K_SUM_TILE, [False] * K_SUM_TILE, [0] * K_SUM_TILE, [0] * K_SUM_TILE
    for tid in range(K_SUM_BLOCK):
        prev = normal_code(float(base[tid]))
        for j in range(K_SUM_PER):
            k = tid * K_SUM_PER + j
            cb[k] = prev
            with np.errstate(all="ignore"):
                ca[k] = normal_code(float(base[tid] + loc[tid, j])) if k < real else prev
            r = _ldexp(x[k], 52 - code_exp(cb[k]))
            ri = float(np.rint(r))
            conv = (cb[k] >= 0 and ca[k] == cb[k] and abs(r) < 9007199254740992.0 and
                    abs(r - ri) != 0.5)
            single[k] = k < real and not conv
            q[k] = int(ri) if conv else 0
            prev = ca[k]
    flag = [single[k] or (k < real and (ca[k - 1] if k else -3) != cb[k])
            for k in range(K_SUM_TILE)]
    count = sum(flag)
    if count > K_ITEM_CAP:
        return None
    start, xs, code, elem = [0] * (K_ITEM_CAP + 1), [0.0] * count, [0] * count, [0] * count
    lo, hi = [LL_MAX] * count, [LL_MIN] * count
    ids, pre, cur = [], 0, -1
    pres = []
    for k in range(K_SUM_TILE):
        if flag[k]:
            cur += 1
            bnd.see("start", cur)
            bnd.see("xn", cur)
            start[cur] = pre
            xs[cur] = float(x[k]) if single[k] else 0.0
            code[cur] = ca[k] if single[k] else cb[k]
            elem[cur] = k + (1 if single[k] else 0)
            bnd.see("lo", cur)
        pre = wrap64(pre + q[k])
        ids.append(cur)
        pres.append(pre)
    bnd.see("start", count)
    start[count] = pre
    for k in range(real):
        if not single[k]:
            bnd.see("lo", ids[k])
            d = wrap64(pres[k] - start[ids[k]])
            lo[ids[k]] = min(lo[ids[k]], d)
            hi[ids[k]] = max(hi[ids[k]], d)
    items = []
    for i in range(count):
        total = wrap64(start[i + 1] - start[i])
        if lo[i] > hi[i]:
            items.append((xs[i], 0.0, lo[i], hi[i], K_ITEM_NONE, elem[i]))
        else:
            items.append((xs[i], _ldexp(float(total), code_exp(code[i]) - 52), max(lo[i], -HUGE),
                          min(hi[i], HUGE), code[i], elem[i]))
        bnd.see("items", b * K_ITEM_CAP + i)
    return items


def run_applies(s, code, lo, hi):
    if not sum_normal(s) or sign_exp(s) != code:
        return False
    S = int(_ldexp(s, 52 - code_exp(code)))
    lo52, hi53 = (1 << 52) + 1, (1 << 53) - 1
    return (S + lo >= lo52 and S + hi <= hi53) if s > 0 else (S + lo >= -hi53 and S + hi <= -lo52)


def walk_tile(s, b, pos, t, n, buf, bnd):
    begin = b * K_SUM_TILE
    length = min(n, begin + K_SUM_TILE) - begin
    if length <= pos:
        return s
    src = begin + np.minimum(np.arange(K_SUM_TILE), length - 1)
    bnd.see("t", src)
    buf[:K_SUM_TILE] = t[src]
    return wave_walk(buf, length, s, bnd, pos)


def chain_items(t, n, items, bnd):
    """The chain over the tiles' items; returns (sum, tiles walked)."""
    nt = sum_tiles(n)
    counts = [len(i) if i is not None else -1 for i in items]
    buf = np.zeros(K_SUM_BUF)
    s, bb, walked = 0.0, 0, 0
    lo52, hi53 = (1 << 52) + 1, (1 << 53) - 1
    while bb < nt and not math.isnan(s):
        k = [bb + lane for lane in range(64)]
        inn = [v < nt for v in k]
        cnt = [counts[v] if v < nt else 0 for v in k]
        bnd.see("counts", [min(v, nt - 1) for v in k])
        f = 0
        if inn[0] and cnt[0] == 1 and sum_normal(s):
            c = sign_exp(s)
            e = code_exp(c)
            S, incl, f = int(_ldexp(s, 52 - e)), 0, 64
            for lane in range(64):
                ok, N = False, 0
                if inn[lane] and cnt[lane] == 1:
                    bnd.see("items", k[lane] * K_ITEM_CAP)
                    x, nd, lo, hi, code, _ = items[k[lane]][0]
                    if x == 0.0 and code == c:
                        N = int(_ldexp(nd, 52 - e))
                        at = S + incl
                        ok = (at + lo >= lo52 and at + hi <= hi53) if s > 0 else \
                            (at + lo >= -hi53 and at + hi <= -lo52)
                if not ok:
                    f = lane
                    break
                incl += N
            if f > 0:
                s = _ldexp(float(S + incl), e - 52)
        if f >= 8 or bb + f >= nt:
            bb += f
            continue
        use = [cnt[lane] if lane >= f and inn[lane] else 0 for lane in range(64)]
        incl = list(np.cumsum([max(u, 0) for u in use]))
        g = 64
        for lane in range(64):
            if not inn[lane] or (lane >= f and (cnt[lane] < 0 or incl[lane] > K_ITEM_WIN)):
                g = lane
                break
        assert g >= f
        if g == f:
            # a tile without items (the kernel relies on a tile's fitting a window)
            assert cnt[f] < 0
            s = walk_tile(s, bb + f, 0, t, n, buf, bnd)
            walked += 1
            bb += f + 1
            continue
        total = int(incl[g - 1])
        at = [int(incl[lane]) - max(use[lane], 0) if lane < g else LL_MAX for lane in range(64)]
        staged = [None] * total
        for q0 in range(0, total, 64 * K_ITEM_PASS):
            for lane in range(64):
                if q0 + lane >= total:
                    continue
                for u in range(K_ITEM_PASS):
                    q = min(q0 + lane + 64 * u, total - 1)
                    li = 0
                    for o in (32, 16, 8, 4, 2, 1):
                        bnd.see("at", li + o)
                        if at[li + o] <= q:
                            li += o
                    bnd.see("items", (bb + li) * K_ITEM_CAP + (q - at[li]))
                    bnd.see("xn", q)
                    bnd.see("lo", q)
                    staged[q] = items[bb + li][q - at[li]]
        bnd.see("xn", total + 7)
        mid = []
        for q0 in range(0, total, 8):
            bnd.see("mid", q0 + 7)
            bnd.see("xn", min(q0 + 15, K_ITEM_WIN + 7))
        with np.errstate(all="ignore"):
            for x, nd, *_ in staged:
                s = float(np.float64(s) + x)
                mid.append(s)
                s = float(np.float64(s) + nd)
        fail = next((i for i, (x, nd, lo, hi, code, _) in enumerate(staged)
                     if code != K_ITEM_NONE and not run_applies(mid[i], code, lo, hi)), -1)
        if fail < 0:
            bb += g
            continue
        s = mid[fail]
        li = next(lane for lane in range(f, g) if cnt[lane] > 0 and at[lane] <= fail < at[lane] + cnt[lane])
        s = walk_tile(s, bb + li, staged[fail][5], t, n, buf, bnd)
        walked += 1
        bb += li + 1
    return s, walked


def emulate(t):
    t = np.asarray(t, dtype=np.float64)
    n, bnd = len(t), Bounds()
    nt = sum_tiles(n)
    with np.errstate(all="ignore"):
        tsum = [float(np.sum(t[b * K_SUM_TILE:(b + 1) * K_SUM_TILE])) for b in range(nt)]
        items = [tile_items(t, n, b, float(np.sum(tsum[:b])), bnd) for b in range(nt)]
    s, walked = chain_items(t, n, items, bnd)
    for name, size in (("t", n), ("counts", nt), ("items", nt * K_ITEM_CAP), ("at", 64),
                       ("start", K_ITEM_CAP + 1), ("xn", K_ITEM_WIN + 8), ("mid", K_ITEM_WIN + 8),
                       ("lo", K_ITEM_WIN), ("buf", K_SUM_BUF)):
        bnd.check(name, size)
    return s, walked, items


def crafted():
    """Inputs whose items go wrong: predictions that miss, tiles with exactly
    as many items as fit and one more, windows filled to their end."""
    rng = np.random.default_rng(2)
    out = {}
    h = rng.choice([-3, -2, -1, 1, 2, 3], 9 * 1024 + 5) * 2.0 ** -53
    h[0] = 1.0
    out["hover"] = h
    c = rng.standard_normal(9 * 1024 + 5) * 10.0 ** np.linspace(60, 20, 9 * 1024 + 5)
    c[1::2] = -c[0::2][: len(c[1::2])] * (1 + 1e-10 * rng.standard_normal(len(c[1::2])))
    out["cancel"] = c
    # a binade change and back every 2 m addends: two items per swing
    for name, swings in (("at the cap", 128), ("past the cap", 129)):
        t = np.zeros(6 * 1024)
        t[0] = 1.5
        for b in range(1, 6):
            at = b * 1024 + 4 * np.arange(swings)
            t[at], t[at + 2] = 1.0, -1.0
        out[name] = t
    out["full windows"] = np.tile(np.where(np.arange(1024) % 8 == 0, 1.0, 0.0) *
                                  np.where(np.arange(1024) % 16 == 0, 1.0, -1.0), 70)
    out["full windows"][0] = 1.5
    return out


@pytest.mark.parametrize("k", range(len(_cases())))
def test_emulated_items_in_bounds_and_exact(k):
    t = _cases()[k]
    if len(t) > 20000:
        t = t[:20000]
    got, _, _ = emulate(t)
    want = _sequential(t)
    assert got == want or (math.isnan(got) and math.isnan(want)), (len(t), got, want)


@pytest.mark.parametrize("name", sorted(crafted()))
def test_emulated_items_where_they_go_wrong(name):
    t = crafted()[name]
    got, walked, items = emulate(t)
    assert got == _sequential(t)
    most = max(len(i) if i is not None else K_ITEM_CAP + 1 for i in items)
    if name == "past the cap":
        assert most > K_ITEM_CAP and walked > 0
    if name == "at the cap":
        assert most == K_ITEM_CAP
    if name == "hover":
        assert walked > 0
