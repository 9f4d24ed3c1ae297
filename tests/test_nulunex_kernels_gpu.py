"""Each mechanism of the Nulunex decoder alone, kernel by kernel: rows of q and k with a norm per head behind the rotation
and keys that are values too, query rows with neighbouring pairs turned, the latent rows put into their pages, the fold
from 32-bit rows, a decode step's fold and rows in one launch, the pages of a prompt from its first position on, the
decode attention over wide latent rows with its value matrix, and the products that end in the clamped swish."""
import math

import pytest
import torch

import plain_nulunex as P

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F64 = torch.float64
BF = torch.bfloat16


def rel(got, ref):
    return float((got.cpu().to(F64) - ref).abs().max()) / max(float(ref.abs().max()), 1e-30)


def planner_for(key, slots=4, pages=60, dtype=torch.float32, context=4096):
    from agave_amd.cache import KVCache
    from agave_amd.engine.step import StepPlanner
    cache = KVCache({0: key}, {}, slots, {key: pages}, dtype, torch.device(DEV), context)
    return cache, StepPlanner(cache, 1000, torch.device(DEV))


def workspace():
    from agave_amd.parts import Workspace
    return Workspace(torch.device(DEV))


def frequencies(base, pairs):
    return torch.tensor([base ** (-2.0 * e / (2 * pairs)) for e in range(pairs)], dtype=F64, device=DEV)


# ---------------------------------------------------------------- q and k with a norm per head
@pytest.mark.parametrize("dtype", [torch.float32, BF])
@pytest.mark.parametrize("H, G, d, rot, vd", [(6, 3, 16, 8, None), (4, 4, 32, 32, None), (5, 1, 48, 20, None), (2, 2, 20, 0, None),
                                              (3, 1, 10, 2, 7), (8, 2, 128, 128, None), (2, 1, 256, 64, 48), (1, 1, 400, 300, None)])
def test_rows_with_a_norm_per_head_behind_the_rotation(dtype, H, G, d, rot, vd):
    """Rows out and rows into the cache pages (either order), 64 rows and more; the values are the keys as they came
    (``vd`` None) or rows of their own; positions on both sides of a page's border and far out."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import attention_biased as A
    own_v = vd is not None
    vd = vd or d
    eps = 3e-4
    for n in (70, 9):
        g = torch.Generator().manual_seed(d + n)
        cache, planner = planner_for(GroupKey(None, G, d, v_head_dim=vd, layout="rows_vt"), dtype=dtype)
        cache.alloc_slot()
        slot = cache.alloc_slot()
        if n == 9:
            ahead = planner.plan([slot], [[0] * 2043], "all")           # the nine rows stand at positions 2,043 and on
            planner.commit(ahead)
        step = planner.plan([slot], [[0] * n], "all")
        wide = torch.randn(n, H * d + G * d + G * vd + 4, generator=g) * 2
        dev = wide.to(DEV)
        q, k = dev[:, :H * d], dev[:, H * d:H * d + G * d]
        v = dev[:, H * d + G * d:H * d + G * d + G * vd] if own_v else None
        freq = frequencies(700.0, rot // 2) if rot else None
        pos = step.tok_pos.cpu().long()
        q64, k64 = wide.to(F64)[:, :H * d].view(n, H, d), wide.to(F64)[:, H * d:H * d + G * d].view(n, G, d)
        v64 = v.cpu().to(F64) if own_v else wide.to(F64)[:, H * d:H * d + G * d]
        turn = (lambda x: P.turn_halves(x, pos, rot, 700.0)) if rot else (lambda x: x)
        want_q, want_k = P.rms(turn(q64), eps).reshape(n, -1), P.rms(turn(k64), eps).reshape(n, -1)
        outs = [torch.empty(n, c, dtype=dtype, device=DEV) for c in (H * d, G * d, G * vd)]
        A.head_norm_rope(q, k, v, *outs, eps, eps, freq, 1.0, step, H, G, d, vd)
        tol = 3e-6 if dtype == torch.float32 else 5e-3
        for got, want, what in zip(outs, (want_q, want_k, v64), "qkv"):
            assert rel(got, want) < tol, (what, n)
        # straight into the pages: the same as the rows appended afterwards
        kp, vp, packed = cache.pages_of(0)
        table, base = step.tables[0]
        q2 = torch.empty_like(outs[0])
        A.head_norm_rope(q, k, v, q2, None, None, eps, eps, freq, 1.0, step, H, G, d, vd, pages=(kp, vp, table, base, 0, packed))
        kp2, vp2 = torch.zeros_like(kp), torch.zeros_like(vp)
        A.kv_append_rows(outs[1], outs[2], kp2, vp2, table, base, 0, step, G, d, vd, packed)
        assert torch.equal(q2, outs[0]) and torch.equal(kp, kp2) and torch.equal(vp, vp2) and float(kp.abs().max()) > 0
        # queries alone (a run that appends nothing), with the sine and cosine of a scaled rotation
        q3 = torch.empty_like(q2)
        A.head_norm_rope(q, None, None, q3, None, None, eps, eps, freq, 1.7, step, H, G, d, vd)
        x = turn(q64)
        scaled = torch.cat([1.7 * x[..., :rot], x[..., rot:]], -1)
        assert rel(q3, P.rms(scaled, eps).reshape(n, -1)) < tol


# ---------------------------------------------------------------- the latent attention's rows
@pytest.mark.parametrize("dtype", [torch.float32, BF])
@pytest.mark.parametrize("heads, dim, rot, kv_rank", [(3, 12, 6, 40), (5, 32, 16, 48), (2, 1, 2, 1), (16, 128, 64, 512)])
def test_query_rows_and_the_cached_row(dtype, heads, dim, rot, kv_rank):
    """Queries straight from a product (32-bit column slices) with neighbouring pairs turned, and the latent row normed
    and turned, as rows and in its place in the pages."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import attention_biased as A
    from agave_amd.ops import latent as L
    n, eps, base, qd, kd = 75, 2e-4, 300.0, dim + rot, kv_rank + rot
    g = torch.Generator().manual_seed(dim)
    cache, planner = planner_for(GroupKey(None, 1, kd, v_head_dim=kv_rank, layout="rows_vt"), dtype=dtype)
    slot = cache.alloc_slot()
    planner.commit(planner.plan([slot], [[0] * 1000], "all"))
    step = planner.plan([slot], [[0] * n], "all")
    wide = torch.randn(n, heads * qd + kd + 3, generator=g) * 2
    w = 1 + 0.3 * torch.randn(kv_rank, generator=g)
    dev = wide.to(DEV)
    q_raw, kv_raw = dev[:, :heads * qd], dev[:, heads * qd:heads * qd + kd]
    turn = L.Turn(frequencies(base, rot // 2), True)
    pos = step.tok_pos.cpu().long()
    q64, r64 = wide.to(F64)[:, :heads * qd].view(n, heads, qd), wide.to(F64)[:, heads * qd:heads * qd + kd]
    want_q = torch.cat([q64[..., :dim], P.turn_neighbours(q64[..., dim:], pos, rot, base)], -1).reshape(n, -1)
    want_row = torch.cat([P.rms(r64[:, :kv_rank], eps) * w.to(F64), P.turn_neighbours(r64[:, None, kv_rank:], pos, rot, base)[:, 0]], -1)
    q, row = torch.empty(n, heads * qd, dtype=dtype, device=DEV), torch.empty(n, kd, dtype=dtype, device=DEV)
    kp, vp, packed = cache.pages_of(0)
    table, tbase = step.tables[0]
    L.latent_prepare(step, eps, turn, rot, q_raw=q_raw, q_out=q, q_heads=heads, q_dim=dim, kv_raw=kv_raw, kv_weight=w.to(DEV), k_row=row,
                     kv_rank=kv_rank, pages=L.CachePages(kp, vp, table, tbase, packed))
    tol = 3e-6 if dtype == torch.float32 else 5e-3
    assert rel(q, want_q) < tol and rel(row[:, :kv_rank], want_row[:, :kv_rank]) < tol and rel(row[:, kv_rank:], want_row[:, kv_rank:]) < tol
    kp2, vp2 = torch.zeros_like(kp), torch.zeros_like(vp)
    A.kv_append_rows(row, row[:, :kv_rank], kp2, vp2, table, tbase, 0, step, 1, kd, kv_rank, packed)
    assert torch.equal(kp, kp2) and torch.equal(vp, vp2) and float(kp.abs().max()) > 0
    # rows already of the activations' type: apart and in place
    typed = q_raw.to(dtype).contiguous()
    apart = torch.empty_like(typed)
    L.turn_queries(typed, apart, heads, dim, rot, turn, step.tok_pos)
    L.turn_queries(typed, typed, heads, dim, rot, turn, step.tok_pos)
    assert torch.equal(typed, apart) and rel(apart, want_q) < 3 * tol


@pytest.mark.parametrize("n", [1, 8, 16, 17, 150])
@pytest.mark.parametrize("heads, dim, rot, kv_rank", [(3, 16, 6, 40), (5, 32, 16, 48), (2, 24, 4, 72), (16, 128, 64, 512), (1, 12, 4, 16)])
def test_fold_of_queries_from_32_bit_rows(n, heads, dim, rot, kv_rank):
    """A bfloat16 step's fold reads the 32-bit rows of the first product (column slices): on the matrix cores and on the
    plain kernel, with neighbouring pairs turned; and up to sixteen tokens the fold and the latent rows in one launch."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import latent as L
    qd, kd, base, eps = dim + rot, kv_rank + rot, 90.0, 1e-5
    g = torch.Generator().manual_seed(n + dim)
    wide = torch.randn(n, (heads * qd + kd + 3) // 4 * 4 + 4, generator=g)
    fold = (torch.randn(heads, kv_rank, dim, generator=g) * dim ** -0.5).to(BF)
    w = 1 + 0.3 * torch.randn(kv_rank, generator=g)
    dev = wide.to(DEV)
    q_raw, kv_raw = dev[:, :heads * qd], dev[:, heads * qd:heads * qd + kd]
    cache, planner = planner_for(GroupKey(None, 1, kd, v_head_dim=kv_rank, layout="rows_vt"), slots=20, pages=40, dtype=BF)
    slots = [cache.alloc_slot() for _ in range(min(n, 16))]
    decode = n <= 16
    if decode:
        planner.commit(planner.plan(slots, [[0] * (60 + i) for i in range(n)], "all"))
        step = planner.plan(slots, [[0]] * n, "all")
    else:
        step = planner.plan(slots[:1], [[0] * n], "all")
    turn = L.Turn(frequencies(base, rot // 2), True)
    q64 = wide.to(F64)[:, :heads * qd].view(n, heads, qd)
    want = torch.cat([torch.einsum("thk,hck->thc", q64[..., :dim], fold.to(F64)),
                      P.turn_neighbours(q64[..., dim:], step.tok_pos.cpu().long(), rot, base)], -1).reshape(n, -1)
    for plain in (True, False):
        y = torch.empty(n, heads * kd, dtype=BF, device=DEV)
        L.heads_product(q_raw, fold.to(DEV), y, heads, qd, kd, tail=rot, turn=turn, tok_pos=step.tok_pos, force_plain=plain)
        assert rel(y, want) < 1e-2, plain
    if decode and L.decode_rows_ok(q_raw, heads, dim, rot):
        kp, vp, packed = cache.pages_of(0)
        table, tbase = step.tables[0]
        pages = L.CachePages(kp, vp, table, tbase, packed)
        y2, row = torch.empty_like(y), torch.empty(n, kd, dtype=BF, device=DEV)
        L.decode_rows(q_raw, fold.to(DEV), y2, heads, dim, rot, turn, kv_raw, w.to(DEV), kv_rank, pages, step, eps)
        kp1, vp1 = kp.clone(), vp.clone()
        kp.zero_()
        vp.zero_()
        L.latent_prepare(step, eps, turn, rot, kv_raw=kv_raw, kv_weight=w.to(DEV), k_row=row, kv_rank=kv_rank, pages=pages)
        assert torch.equal(y, y2) and torch.equal(kp, kp1) and torch.equal(vp, vp1) and float(kp1.abs().max()) > 0
    else:
        assert n > 16 or dim % 8 or (dim + rot) % 4


@pytest.mark.parametrize("heads, dim, rot, vd, kv_rank", [(3, 16, 8, 16, 40), (5, 32, 16, 48, 64), (16, 128, 64, 128, 512), (2, 8, 0, 32, 8)])
def test_pages_of_a_prompt_from_its_first_position(heads, dim, rot, vd, kv_rank):
    """Keys and values of every head into pages that hold rubbish before: the same as the rows appended one by one to
    pages of zeros, for sequences of a page, of less, of more, and of one token."""
    from agave_amd.ops import attention_biased as A
    from agave_amd.ops import latent as L
    lens, qd = [64, 1, 130, 37, 192], dim + rot
    n, counts = sum(lens), [-(-x // 64) for x in lens]
    g = torch.Generator().manual_seed(vd)
    up = torch.randn(n, heads * (dim + vd), generator=g).to(BF).to(DEV)
    row = torch.randn(n, kv_rank + rot, generator=g).to(BF).to(DEV)
    table = torch.zeros(len(lens), max(counts), dtype=torch.int32)
    at = 0
    order = torch.randperm(sum(counts), generator=g).to(torch.int32)             # pages in no order
    for b, c in enumerate(counts):
        table[b, :c] = order[at:at + c]
        at += c
    table = table.to(DEV)

    class Step:
        n_tokens, n_seqs = n, len(lens)
        cu = [sum(lens[:i]) for i in range(len(lens) + 1)]
        cu_dev = torch.tensor(cu, dtype=torch.int32, device=DEV)
        tok_seq = torch.tensor([b for b, x in enumerate(lens) for _ in range(x)], dtype=torch.int32, device=DEV)
        tok_pos = torch.tensor([t for x in lens for t in range(x)], dtype=torch.int32, device=DEV)
    hd_k = (qd + 31) // 32 * 32
    kp = torch.full((at, heads, 64, hd_k), 7.5, dtype=BF, device=DEV)
    vp = torch.full((at, heads, vd, 64), float("nan"), dtype=BF, device=DEV)
    L.fresh_pages(up, row, kv_rank, kp, vp, table, Step, heads, dim, rot, vd)
    k = torch.cat([up[:, :heads * dim].view(n, heads, dim), row[:, None, kv_rank:].expand(n, heads, rot)], -1).reshape(n, -1).contiguous()
    v = up[:, heads * dim:].contiguous()
    kp2, vp2 = torch.zeros_like(kp), torch.zeros(vp.shape, dtype=BF, device=DEV)
    base = torch.zeros(len(lens), dtype=torch.int32, device=DEV)
    A.kv_append_rows(k, v, kp2, vp2, table, base, 0, Step, heads, qd, vd, True)
    assert torch.equal(kp, kp2) and torch.equal(vp, vp2)


# ---------------------------------------------------------------- decode attention over latent rows
def plain_decode(q, rows, scale, window, sink, v_up, gate, pos):
    """One query row [heads, kd] at position ``pos`` over rows [pos + 1, kd]."""
    lo = max(0, pos - window + 1) if window else 0
    kv = rows[lo:pos + 1]
    out = []
    for h in range(q.shape[0]):
        s = (kv @ q[h]) * scale
        top = max(float(s.max()), float(sink[h]) if sink is not None else -math.inf)
        p = torch.exp(s - top)
        z = p.sum() + (math.exp(float(sink[h]) - top) if sink is not None else 0.0)
        out.append(v_up[h] @ ((p / z) @ kv[:, :v_up.shape[2]]))
    y = torch.stack(out).reshape(-1)
    return y * torch.sigmoid(gate) if gate is not None else y


@pytest.mark.parametrize("heads, kd, kv_rank, out, window, with_sink, with_gate", [
    (4, 40, 32, 16, 70, True, False),           # less than one step of elements in a wave's half, a window over a page's border
    (1, 24, 16, 10, None, False, True),         # one head, one step, outputs that are no multiple of 16
    (20, 144, 112, 24, 64, True, True),         # two groups of heads, a window of exactly a page
    (16, 576, 512, 128, 300, True, False),      # the widest rows
    (33, 320, 272, 200, None, True, False),     # three groups of heads, sizes between the kernel's own
    (3, 64, 48, 8, 1, True, False),             # a window of the token itself
    (2, 200, 144, 40, 129, False, False)])
@pytest.mark.parametrize("splits", [None, 1, 3, 64])
def test_decode_attention_over_latent_rows(heads, kd, kv_rank, out, window, with_sink, with_gate, splits):
    """Sequences of several lengths in one step (first position, a page's last and first place, many pages), a page
    shared out among one to 64 workgroups (more than there are pages)."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import attention_biased as A
    from agave_amd.ops import latent as L
    before = [0, 63, 64, 130, 777]
    g = torch.Generator().manual_seed(kd + heads)
    cache, planner = planner_for(GroupKey(window, 1, kd, v_head_dim=kv_rank, layout="rows_vt"), slots=5, pages=60, dtype=BF)
    slots = [cache.alloc_slot() for _ in before]
    rows = [torch.randn(n + 1, kd, generator=g).to(BF) for n in before]
    v_up = (torch.randn(heads, out, kv_rank, generator=g) * kv_rank ** -0.5).to(BF)
    sink = torch.randn(heads, generator=g) * 2 if with_sink else None
    kp, vp, packed = cache.pages_of(0)
    assert packed and L.decode_attention_ok(kd, kv_rank, out)

    def append(step, r):
        r = r.to(DEV)
        table, base = step.tables[0]
        A.kv_append_rows(r, r[:, :kv_rank], kp, vp, table, base, 0, step, 1, kd, kv_rank, packed)
    some = [i for i, n in enumerate(before) if n]
    step = planner.plan([slots[i] for i in some], [[0] * before[i] for i in some], "all")
    append(step, torch.cat([rows[i][:-1] for i in some]))
    planner.commit(step)
    step = planner.plan(slots, [[0]] * len(before), "all")
    append(step, torch.stack([r[-1] for r in rows]))
    q = (torch.randn(len(before), heads * kd, generator=g) * 1.5).to(BF)
    gate = torch.randn(len(before), heads * out + 3, generator=g) if with_gate else None
    y = torch.full((len(before), heads * out), 9.0, dtype=BF, device=DEV)
    table, base = step.tables[0]
    scale = 0.8 * kd ** -0.5
    L.decode_attention(q.to(DEV), v_up.to(DEV), y, gate.to(DEV)[:, 2:2 + heads * out] if with_gate else None, kp, vp, table, base, step,
                       heads, kd, kv_rank, scale, window, sink.to(DEV) if with_sink else None, workspace(), splits=splits)
    want = torch.stack([plain_decode(q[i].to(F64).view(heads, kd), rows[i].to(F64), scale, window, sink, v_up.to(F64),
                                     gate[i, 2:2 + heads * out].to(F64) if with_gate else None, before[i]) for i in range(len(before))])
    for i in range(len(before)):
        assert rel(y[i], want[i]) < 1.5e-2, (before[i], rel(y[i], want[i]))


@pytest.mark.parametrize("splits", [1, 3, 64])
@pytest.mark.parametrize("window", [None, 4200])
def test_decode_attention_over_tables_of_more_columns_than_a_wave_has_lanes(window, splits):
    """Sequences of one page, of 64, of 65 and of 130, with and without pages that a table does not name: a share's first page is
    named by a lane among the first 64 columns, the others by loads of their own.  Queries, weights and the merged row are rounded to bfloat16 (2^-9 each), the result too."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import attention_biased as A
    from agave_amd.ops import latent as L
    heads, kd, kv_rank, out, before = 3, 40, 32, 16, [40, 4095, 4096, 8300]
    g = torch.Generator().manual_seed(splits)
    cache, planner = planner_for(GroupKey(window, 1, kd, v_head_dim=kv_rank, layout="rows_vt"), slots=4, pages=280, dtype=BF, context=9000)
    slots, rows = [cache.alloc_slot() for _ in before], [torch.randn(n + 1, kd, generator=g).to(BF) for n in before]
    v_up = (torch.randn(heads, out, kv_rank, generator=g) * kv_rank ** -0.5).to(BF)
    kp, vp, packed = cache.pages_of(0)
    for lo in range(0, 8301, 1000):
        some = [i for i, n in enumerate(before) if n > lo]
        part = [rows[i][lo:min(lo + 1000, before[i])] for i in some]
        step = planner.plan([slots[i] for i in some], [[0] * len(r) for r in part], "all")
        r, (table, base) = torch.cat(part).to(DEV), step.tables[0]
        A.kv_append_rows(r, r[:, :kv_rank], kp, vp, table, base, 0, step, 1, kd, kv_rank, packed)
        planner.commit(step)
    step = planner.plan(slots, [[0]] * len(before), "all")
    table, base = step.tables[0]
    r = torch.stack([x[-1] for x in rows]).to(DEV)
    A.kv_append_rows(r, r[:, :kv_rank], kp, vp, table, base, 0, step, 1, kd, kv_rank, packed)
    q, first = torch.randn(len(before), heads * kd, generator=g).to(BF), base.cpu().tolist()
    for gone in ((), (70, 71, 128, 129)):
        held = table.clone()
        for page in gone:
            held[3, page - first[3]] = -1
        y = torch.empty(len(before), heads * out, dtype=BF, device=DEV)
        L.decode_attention(q.to(DEV), v_up.to(DEV), y, None, kp, vp, held, base, step, heads, kd, kv_rank, kd ** -0.5, window, None, workspace(),
                           splits=splits)
        for i, n in enumerate(before):
            lo = max(0, n - window + 1) if window else 0
            kept = torch.tensor([p for p in range(lo, n + 1) if i < 3 or p // 64 not in gone])
            want = plain_decode(q[i].to(F64).view(heads, kd), rows[i][kept].to(F64), kd ** -0.5, None, None, v_up.to(F64), None, len(kept) - 1)
            assert rel(y[i], want) < 1.5e-2, (n, gone)


def test_a_growing_sequence_moves_no_buffer_of_latent_attention():
    """More pages, more shares of a row: their results lie in the buffers that the first step has made, so that steps that were recorded
    with their addresses stay valid."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import attention_biased as A
    from agave_amd.ops import latent as L
    heads, kd, kv_rank, out, T = 16, 40, 32, 16, 1400
    g = torch.Generator().manual_seed(3)
    cache, planner = planner_for(GroupKey(None, 1, kd, v_head_dim=kv_rank, layout="rows_vt"), slots=1, pages=30, dtype=BF)
    slot, ws, rows = cache.alloc_slot(), workspace(), torch.randn(T, kd, generator=g).to(BF)
    v_up = (torch.randn(heads, out, kv_rank, generator=g) * kv_rank ** -0.5).to(BF)
    kp, vp, packed = cache.pages_of(0)
    planner.fixed_width, at = [64], 0
    for n in (9, 1, 60, 1, 300, 1, T - 373, 1):
        step = planner.plan([slot], [[0] * n], "all")
        r, (table, base) = rows[at:at + n].to(DEV), step.tables[0]
        A.kv_append_rows(r, r[:, :kv_rank], kp, vp, table, base, 0, step, 1, kd, kv_rank, packed)
        if n == 1:
            q, y = torch.randn(1, heads * kd, generator=g).to(BF), torch.empty(1, heads * out, dtype=BF, device=DEV)
            L.decode_attention(q.to(DEV), v_up.to(DEV), y, None, kp, vp, table, base, step, heads, kd, kv_rank, kd ** -0.5, None, None, ws)
            want = plain_decode(q.to(F64).view(heads, kd), rows.to(F64), kd ** -0.5, None, None, v_up.to(F64), None, at)
            assert rel(y[0], want) < 1.5e-2, at
        planner.commit(step)
        at += n
    assert ws.generation == 0 and ws.allocations == 2


@pytest.mark.parametrize("splits", [1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("rows, heads, vd, out", [(1, 2, 48, 10), (3, 20, 256, 40), (9, 16, 512, 128), (17, 16, 272, 200)])
def test_latent_shares_merged_and_multiplied(rows, heads, vd, out, splits):
    """One to eight workgroups a (row, head), every number of shares a group of threads keeps, shares without a key.  The merged row is
    rounded to bfloat16, the product's result too: half a unit in the last of eight places each."""
    from agave_amd.ops import latent as L
    from agave_amd.ops import library
    from agave_amd.ops.kernels import ptr, stream
    g = torch.Generator().manual_seed(splits + out)
    part = torch.randn(rows, heads, splits, vd, generator=g)
    ml = torch.stack([torch.randn(rows, heads, splits, generator=g) * 3, torch.rand(rows, heads, splits, generator=g) + 0.5], -1)
    empty = torch.rand(rows, heads, splits, generator=g) < 0.3
    empty[..., 0] = False
    ml[..., 0][empty], ml[..., 1][empty], part[empty] = float("-inf"), 0.0, 0.0
    w, gate = (torch.randn(heads, out, vd, generator=g) * vd ** -0.5).to(BF), torch.randn(rows, heads * out, generator=g)
    y = torch.full((rows, heads * out + 3), 9.0, dtype=BF, device=DEV)
    d = [t.to(DEV) for t in (part, ml, w, gate)]
    library.call(L._attn(), "agave_latent_values", ptr(d[0]), ptr(d[1]), splits, ptr(d[2]), ptr(y), y.stride(0), ptr(d[3]), heads * out, rows, heads,
                 vd, out, stream())
    f = torch.exp2(ml[..., 0].to(F64) - ml[..., 0].to(F64).amax(-1, keepdim=True))
    merged = (part.to(F64) * f[..., None]).sum(2) / (f * ml[..., 1].to(F64)).sum(-1)[..., None]
    turned, opened = torch.einsum("rhd,hod->rho", merged, w.to(F64)), torch.sigmoid(gate.to(F64)).view(rows, heads, out)
    most = torch.einsum("rhd,hod->rho", merged.abs(), w.to(F64).abs()) * opened
    want = turned * opened
    got = y[:, :heads * out].cpu().to(F64).view(rows, heads, out)
    assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + (2.0 ** -9 + 2.0 ** -16) * most).all())
    assert bool((y[:, heads * out:] == 9.0).all())


@pytest.mark.parametrize("n", [1, 16, 17])
@pytest.mark.parametrize("heads", [1, 64, 65])
def test_folds_of_few_tokens(n, heads):
    """16 or 64 columns a wave, turned elements from workgroups of their own: up to 512 workgroups and beyond, the largest step of few
    tokens and the next.  Queries are rounded to bfloat16 on the way in, the result too."""
    from agave_amd.ops import latent as L
    K, n_out, rot = 40, 500, 8
    g = torch.Generator().manual_seed(n + heads)
    x, w = torch.randn(n, heads * (K + rot), generator=g), (torch.randn(heads, n_out, K, generator=g) * K ** -0.5).to(BF)
    freq = torch.rand(rot // 2, generator=g).to(F64)
    pos = torch.arange(n, dtype=torch.int32) * 7
    y = torch.full((n, heads * (n_out + rot)), float("nan"), dtype=BF, device=DEV)
    L.heads_product(x.to(DEV), w.to(DEV), y, heads, K + rot, n_out + rot, tail=rot, turn=L.Turn(freq.to(DEV)), tok_pos=pos.to(DEV))
    got, x = y.cpu().to(F64).view(n, heads, -1), x.to(F64).view(n, heads, -1)
    want, most = (torch.einsum("nhk,hok->nho", v, u) for v, u in ((x[..., :K], w.to(F64)), (x[..., :K].abs(), w.to(F64).abs())))
    assert bool(((got[..., :n_out] - want).abs() <= 2.0 ** -8 * want.abs() + (2.0 ** -9 + 2.0 ** -16) * most).all())
    angle = pos.to(F64)[:, None, None] * freq
    a, b = x[..., K:K + rot // 2], x[..., K + rot // 2:]
    turned = torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)
    assert bool(((got[..., n_out:] - turned).abs() <= 2.0 ** -8 * turned.abs() + 2.0 ** -20 * (a.abs() + b.abs()).repeat(1, 1, 2)).all())


@pytest.mark.parametrize("window", [5, 64, 65, 200])
def test_a_key_at_the_windows_edge_of_the_decode_attention(window):
    """One row stands out by thirty in the score, just inside and just outside the window, at page borders and at the
    query's own place: its values fill the result or are absent."""
    from agave_amd.cache import GroupKey
    from agave_amd.ops import attention_biased as A
    from agave_amd.ops import latent as L
    kd, kv_rank, heads, n = 48, 32, 2, 400
    for last in (n - 1, 319, 320):
        for at in {last - window + 1, last - window, last, max(0, last // 64 * 64 - 1), last // 64 * 64, 0}:
            g = torch.Generator().manual_seed(at)
            cache, planner = planner_for(GroupKey(window, 1, kd, v_head_dim=kv_rank, layout="rows_vt"), slots=1, pages=20, dtype=BF)
            slot = cache.alloc_slot()
            rows = 0.1 * torch.randn(last + 1, kd, generator=g)
            rows[:, kd - 1] = 0.0
            rows[at, kd - 1] = 30.0
            rows[at, :kv_rank] = 5.0
            rows = rows.to(BF)
            q = torch.zeros(1, heads * kd)
            q[0, kd - 1::kd] = 1.0
            kp, vp, packed = cache.pages_of(0)
            for lo, hi in ((0, last), (last, last + 1)):
                step = planner.plan([slot], [[0] * (hi - lo)], "all")
                r = rows[lo:hi].to(DEV)
                table, base = step.tables[0]
                A.kv_append_rows(r, r[:, :kv_rank], kp, vp, table, base, 0, step, 1, kd, kv_rank, packed)
                if hi <= last:
                    planner.commit(step)
            y = torch.empty(1, heads * kv_rank, dtype=BF, device=DEV)
            eye = torch.eye(kv_rank).to(BF).expand(heads, kv_rank, kv_rank).contiguous().to(DEV)
            table, base = step.tables[0]
            L.decode_attention(q.to(BF).to(DEV), eye, y, None, kp, vp, table, base, step, heads, kd, kv_rank, 1.0, window, None, workspace())
            seen = last - window < at <= last
            assert (float(y.float().min()) > 4.9) if seen else (float(y.float().abs().max()) < 1.0), (last, at)


# ---------------------------------------------------------------- products that end in a gate's form
@pytest.mark.parametrize("m", [1, 5, 40, 64, 65, 300])
@pytest.mark.parametrize("ff, k", [(24, 40), (200, 96), (512, 256)])
def test_products_that_end_in_the_clamped_swish(m, ff, k):
    """Skinny and tiled products, every tile shape, and the product that makes its normalised row itself; gates and up
    values far outside the limit on both sides."""
    from agave_amd.ops import gemm_mfma as G
    g = torch.Generator().manual_seed(m + ff)
    limit, alpha = 1.3, 1.702
    w = (torch.randn(2 * ff, k, generator=g) * 4 * k ** -0.5).to(BF)
    x = torch.randn(m, k, generator=g).to(BF)
    z = x.to(F64) @ w.to(F64).T
    want = {"swish_clamped": P.clamped_swish(z[:, :ff], z[:, ff:], limit), "silu": z[:, :ff] * torch.sigmoid(z[:, :ff]) * z[:, ff:]}
    assert float(z.abs().max()) > 3 * limit
    packed = G.pack_weight(w.to(DEV), interleave_ff=ff)
    for act, ref in want.items():
        form = G.gate_form_of(act, limit, alpha)
        out = torch.empty(m, ff, dtype=BF, device=DEV)
        G.product(x.to(DEV), packed, out, ff, epilogue=1, form=form)
        assert rel(out, ref) < 5e-3, act
        if m > 64:
            for tile in range(4):
                out.fill_(9.0)
                G.tiled_as(x.to(DEV), packed, out, ff, tile, epilogue=1, form=form)
                assert rel(out, ref) < 5e-3, (act, tile)
        if m == 1:
            h = torch.randn(1, k, generator=g)
            gain = 1 + 0.2 * torch.randn(k, generator=g)
            out1 = torch.empty(1, ff, dtype=BF, device=DEV)
            G.row_normed(h.to(DEV), None, None, None, 0.0, gain.to(DEV), 1e-5, packed, out1, ff, epilogue=1, form=form)
            xn = (P.rms(h.to(F64), 1e-5) * gain.to(F64)).to(BF).to(F64)
            zn = xn @ w.to(F64).T
            rn = P.clamped_swish(zn[:, :ff], zn[:, ff:], limit) if act == "swish_clamped" else zn[:, :ff] * torch.sigmoid(zn[:, :ff]) * zn[:, ff:]
            assert rel(out1, rn) < 2e-2, act
    assert G.gate_form_of("relu") is None and G.gate_form_of("gelu_tanh") == G.GELU_TANH
