"""The tree parser's reading of a pair table, restated: how alpacc_create decides whether a grammar
takes it (build_tree_tables in alpacc_amd/csrc/alpacc_hip.hip) and what it makes of every entry."""
import numpy as np

LEFT = 0x8000


def entries(px):
    """[(pops, pushes, filled, owners, kind)] of every pair entry, or None when the grammar keeps the
    element-level kernels: pops and pushes are symbols, filled[r] the production that fills pop r
    (-1: none), owners[l] the production that pushes symbol l (-1: none), kind 1 / 2 the entries of
    the start / end terminal."""
    out = []
    for s0, s1, p0, p1 in np.asarray(px.pair_entry).reshape(-1, 4).tolist():
        st = [int(x) for x in px.stacks[s0:s1]]
        pops = 0
        while pops < len(st) and not st[pops] & LEFT:
            pops += 1
        pushes = len(st) - pops
        if any(not x & LEFT for x in st[pops:]) or p1 - p0 > 7 or pops > 8 or pushes > 8:
            return None
        opened, filled = [], []
        owner = [-1] * (p1 - p0)
        for j, pr in enumerate(px.productions[p0:p1].tolist()):
            if opened:
                owner[j] = opened.pop()
            elif len(filled) == pops:
                return None
            else:
                filled.append(j)
            opened += [j] * int(px.arities[pr])
        kind = 0
        if p1 == p0 and pops == 0 and pushes > 0:
            kind, opened = 1, [-1] * pushes
        elif pushes == 0 and not opened and len(filled) < pops:
            kind = 2
        elif len(filled) != pops or len(opened) != pushes:
            return None
        filled += [-1] * (pops - len(filled))
        out.append(([x & 0x7FFF for x in st[:pops]], [x & 0x7FFF for x in st[pops:]], filled, opened,
                    kind, owner))
    return out


def form(px):
    """'rows', 'loops' (the tree parser's two forms) or 'elements'."""
    e = entries(px)
    if e is None:
        return "elements"
    most = max(1, *(len(x[5]) for x in e))
    pops, pushes = max(1, *(len(x[0]) for x in e)), max(1, *(len(x[1]) for x in e))
    slots = 8
    while slots < 4 * pushes:
        slots *= 2
    wave = 4 * (256 * most + 4 + 64 * (slots + 1) + 256 * pops)
    if wave + 4096 > 65536:
        return "elements"
    return "rows" if pops <= 3 and pushes <= 4 and most <= 4 else "loops"


def key_entries(px, kinds):
    """Pair entry of every position of [start] ++ kinds ++ [end]; None when a key has none."""
    q, k, nt = px.q, px.k, px.num_terminals
    w = ([px.empty_terminal] * q + [px.start_terminal] + list(kinds) + [px.end_terminal] +
         [px.empty_terminal] * (k - 1))
    if not px.pair_index.shape[0]:
        return None
    out = []
    for p in range(len(kinds) + 2):
        di = 0
        for t in w[p:p + q + k]:
            di = di * nt + int(t)
        e = int(px.pair_index[di])
        if e == 0xFFFFFFFF:
            return None
        out.append(e)
    return out


def parents(px, kinds):
    """Parents by one stack of owners, or None when the tokens are rejected."""
    table = entries(px)
    ents = key_entries(px, kinds)
    if ents is None:
        return None
    stack, par = [], []
    for e in ents:
        pops, pushes, filled, owners, _, owner = table[e]
        base = len(par)
        par += [base + o if o >= 0 else None for o in owner]
        for sym, j in zip(pops, filled):
            if not stack or stack[-1][0] != sym:
                return None
            _, own = stack.pop()
            if j >= 0:
                par[base + j] = 0 if own < 0 else own
        for sym, o in zip(pushes, owners):
            stack.append((sym, -1 if o < 0 else base + o))
    return par if not stack else None
