"""Each HIP kernel alone against its plain reference, at other sizes than the engine's tiny
models use, in 32-bit and in bfloat16, with inputs made so that a fault shows (a far key that
must win, a window's edge, scattered page ids)."""
import math
import os

import numpy as np
import pytest
import torch

import plain_gemma3 as P

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
DEV = "cuda:0"


def _g(name):
    path = os.path.join(GOLDEN, name + ".bin")
    if not os.path.isfile(path):
        pytest.skip("reference golden vectors not mounted")
    return torch.from_numpy(np.fromfile(path, dtype="<f4").copy())


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def _tol(dtype):
    return dict(atol=2e-6, rtol=2e-6) if dtype == torch.float32 else dict(atol=1e-2, rtol=1e-2)


@pytest.fixture(scope="module")
def K():
    from agave_amd.ops import kernels
    return kernels


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embed_scale(K, dtype):
    table = (torch.randn(300, 72) * 0.05).to(dtype)
    toks = [0, 299, 17, 17, 123]
    out = torch.empty(5, 72, dtype=torch.float32, device=DEV)
    K.embed_scale(_i32(toks), table.to(DEV), math.sqrt(72.0), out)
    ref = P.embed(toks, table.double(), 72)
    assert torch.allclose(out.cpu().double(), ref, atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("e", [100, 2560, 3136])
def test_residual_norm(K, dtype, e):
    n = 7
    h = torch.randn(n, e) * 3
    br = (torch.randn(n, e) * 0.3).to(dtype)
    gp, gq = torch.randn(e) * 0.1 + 1, torch.randn(e) * 0.1 + 1
    hd = h.clone().to(DEV)
    out = torch.empty(n, e, dtype=dtype, device=DEV)
    K.residual_norm(hd, br.to(DEV), gp.to(DEV), 1e-5, out, gq.to(DEV), 3e-6)
    h_ref = h.double() + P.rms_norm(br.double(), gp.double(), 1e-5, add_one=False)
    o_ref = P.rms_norm(h_ref, gq.double(), 3e-6, add_one=False)
    assert torch.allclose(hd.cpu().double(), h_ref, atol=3e-6, rtol=1e-6)      # the sum is 32-bit in both types
    assert torch.allclose(out.cpu().double(), o_ref, **_tol(dtype))
    # norm only, on gathered rows; and a plain add without a norm on the branch
    rows = _i32([5, 0, 5])
    out2 = torch.empty(3, e, dtype=dtype, device=DEV)
    K.residual_norm(hd, None, None, 0.0, out2, gq.to(DEV), 3e-6, rows)
    assert torch.allclose(out2.cpu().double(), o_ref[[5, 0, 5]], **_tol(dtype))
    h3 = h.clone().to(DEV)
    K.residual_norm(h3, br.to(DEV), None, 0.0, None, None, 0.0)
    assert torch.allclose(h3.cpu().double(), h.double() + br.double(), atol=1e-6)

def _inv_rms_bits(x, eps, threads, first=1):
    """1 / rms of every row as the kernel of 16-byte loads makes it, bit by bit: a thread's four squares in fused steps behind the square of
    the ``first`` one (x first would round another of them), its pieces added up, a wave's lanes in pairs 1, 2, 4 .. 32 apart, the waves in
    turn.  (A fused step is made in numpy's long double: a product of 24 by 24 bits is exact there.)"""
    n, e = x.shape
    v = np.zeros((n, -(-e // (4 * threads)) * threads * 4), np.float32)
    v[:, :e] = x
    v = v.reshape(n, -1, threads, 4)
    fma = lambda a, c: (a.astype(np.longdouble) * a + c).astype(np.float32)
    sq = fma(v[..., 3], fma(v[..., 2], fma(v[..., 1 - first], v[..., first] * v[..., first])))
    ss = sq[:, 0]
    for k in range(1, sq.shape[1]):
        ss = ss + sq[:, k]
    ss = ss.reshape(n, threads // 64, 64)
    while ss.shape[-1] > 1:
        ss = ss[..., 0::2] + ss[..., 1::2]
    total = np.zeros(n, np.float32)
    for w in range(threads // 64):
        total = total + ss[:, w, 0]
    return np.float32(1) / np.sqrt(total / np.float32(e) + np.float32(eps))


@pytest.mark.parametrize("n, e, threads", [(64, 1000, 256), (64, 2048, 512), (64, 2560, 640), (65, 2560, 320), (65, 7000, 896), (64, 16384, 1024)])
def test_norms_add_squares_in_one_order(K, n, e, threads):
    """A row's bits come from its elements alone, not from what else a kernel does with it: the same order of roundings in every form
    (a row normed, a branch normed on its way into the stream, the norm of a sum), whatever the compiler fuses around it."""
    g = torch.Generator().manual_seed(e)
    x, gain, eps = torch.randn(n, e, generator=g) * 3, 1 + 0.3 * torch.randn(e, generator=g), 1e-5
    inv = _inv_rms_bits(x.numpy(), eps, threads)
    assert (inv != _inv_rms_bits(x.numpy(), eps, threads, first=0)).any()             # (the order shows in these rows)
    inv, w = torch.from_numpy(inv)[:, None], gain.to(DEV)
    out = torch.empty(n, e, device=DEV)
    K.residual_norm(x.to(DEV), None, None, 0.0, out, w, eps)
    assert torch.equal(out.cpu(), x * inv * gain)
    for parts in (x.to(DEV), torch.stack([x, torch.zeros_like(x)]).to(DEV)):          # as a row, and as slices
        h = torch.zeros(n, e, device=DEV)
        K.residual_norm(h, parts, w, eps, out, w, eps)
        assert torch.equal(h.cpu(), x * inv * gain)
        second = torch.from_numpy(_inv_rms_bits(h.cpu().numpy(), eps, threads))[:, None]
        assert torch.equal(out.cpu(), h.cpu() * second * gain)
        h = torch.zeros(n, e, device=DEV)
        K.norm_of_sum(h, parts, 1.0, None, w, eps, out, w, eps)
        assert torch.equal(h.cpu(), x * (inv * gain))
        second = torch.from_numpy(_inv_rms_bits(h.cpu().numpy(), eps, threads))[:, None]
        assert torch.equal(out.cpu(), h.cpu() * second * gain)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("e", [100, 2560, 20000])
def test_residual_norm_reads_the_stream_elsewhere(K, dtype, e):
    """``src``: the residual rows are read from another tensor and written to h, with a branch, with
    slices, with a norm only and with nothing else to do (both kernels: 20,000 columns are too many
    for the one that holds a row in registers)."""
    n = 4
    src = torch.randn(n, e) * 3
    br = (torch.randn(n, e) * 0.3).to(dtype)
    parts = torch.randn(3, n, e) * 0.3
    gp, gq = torch.randn(e) * 0.1 + 1, torch.randn(e) * 0.1 + 1
    for branch, b_sum in ((br, br.double()), (parts, parts.double().sum(0)), (None, None)):
        h = torch.full((n, e), 9.0, device=DEV)
        s_dev = src.clone().to(DEV)
        out = torch.empty(n, e, dtype=dtype, device=DEV)
        K.residual_norm(h, branch.to(DEV) if branch is not None else None, gp.to(DEV) if branch is not None else None, 1e-5,
                        out, gq.to(DEV), 3e-6, src=s_dev)
        h_ref = src.double() + (P.rms_norm(b_sum, gp.double(), 1e-5, add_one=False) if b_sum is not None else 0.0)
        assert torch.allclose(h.cpu().double(), h_ref, atol=3e-6, rtol=1e-6)
        assert torch.allclose(out.cpu().double(), P.rms_norm(h_ref, gq.double(), 3e-6, add_one=False), **_tol(dtype))
        assert torch.equal(s_dev.cpu(), src)
    h = torch.full((n, e), 9.0, device=DEV)
    K.residual_norm(h, br.to(DEV), None, 0.0, None, None, 0.0, src=src.to(DEV))         # a plain add
    assert torch.allclose(h.cpu().double(), src.double() + br.double(), atol=1e-6)
    K.residual_norm(h, None, None, 0.0, None, None, 0.0, src=src.to(DEV))               # nothing but the move
    assert torch.equal(h.cpu(), src)
    with pytest.raises(ValueError):
        K.residual_norm(h, None, None, 0.0, None, None, 0.0, src=h)
    with pytest.raises(ValueError):
        K.residual_norm(h, None, None, 0.0, torch.empty(1, e, dtype=dtype, device=DEV), gq.to(DEV), 1e-6, _i32([1]), src=src.to(DEV))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("e", [72, 2560, 5000])
def test_residual_norm_takes_a_branch_in_slices(K, dtype, e):
    """A float32 [slices, rows, hidden] branch stands for the sum of its slices: the same residual
    stream and output as with the sum given as one 32-bit branch (both row-in-registers and plain kernel)."""
    n, slices = 5, 3
    h = torch.randn(n, e) * 3
    parts = torch.randn(slices, n, e) * 0.3
    gp, gq = torch.randn(e) * 0.1 + 1, torch.randn(e) * 0.1 + 1
    hd = h.clone().to(DEV)
    out = torch.empty(n, e, dtype=dtype, device=DEV)
    K.residual_norm(hd, parts.to(DEV), gp.to(DEV), 1e-5, out, gq.to(DEV), 3e-6)
    h_ref = h.double() + P.rms_norm(parts.double().sum(0), gp.double(), 1e-5, add_one=False)
    o_ref = P.rms_norm(h_ref, gq.double(), 3e-6, add_one=False)
    assert torch.allclose(hd.cpu().double(), h_ref, atol=3e-6, rtol=1e-6)
    assert torch.allclose(out.cpu().double(), o_ref, **_tol(dtype))
    h3 = h.clone().to(DEV)
    K.residual_norm(h3, parts.to(DEV), None, 0.0, None, None, 0.0)           # a plain add of the slices
    assert torch.allclose(h3.cpu().double(), h.double() + parts.double().sum(0), atol=2e-6)
    with pytest.raises(ValueError):
        K.residual_norm(h3, parts[:, :4].to(DEV), None, 0.0, None, None, 0.0)


@pytest.mark.parametrize("n", [128, 1152, 2560, 3136])
def test_residual_norm_golden(K, n):
    # research/kernels/generate_golden.py:98-110 (eps 1e-5, plain weight)
    x, w, want = _g(f"rms_norm_n{n}_x"), _g(f"rms_norm_n{n}_w"), _g(f"rms_norm_n{n}_out")
    h = x.view(1, n).clone().to(DEV)
    out = torch.empty(1, n, dtype=torch.float32, device=DEV)
    K.residual_norm(h, None, None, 0.0, out, w.to(DEV), 1e-5)
    assert torch.allclose(out.cpu().view(-1), want, atol=2e-5, rtol=1e-5)


def _pages(n_pages, nkv, hd, dtype):
    k = torch.zeros(n_pages, nkv, 64, hd, dtype=dtype, device=DEV)
    v = torch.zeros(n_pages, nkv, hd, 64, dtype=dtype, device=DEV)
    return k, v


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_qk_norm_rope_kv(K, dtype):
    nh, nkv, hd, rot = 3, 1, 40, 24           # head size no multiple of 16, partial rotation
    seqs = [(0, 5, 3), (1, 130, 4)]           # (sequence, first position, tokens)
    tok_seq = [b for b, _, n in seqs for _ in range(n)]
    tok_pos = [p + i for _, p, n in seqs for i in range(n)]
    n = len(tok_pos)
    q = (torch.randn(n, nh * hd)).to(dtype)
    k = (torch.randn(n, nkv * hd)).to(dtype)
    v = (torch.randn(n, nkv * hd)).to(dtype)
    qg, kg = torch.randn(hd) * 0.1 + 1, torch.randn(hd) * 0.1 + 1
    inv = torch.from_numpy(np.exp(-np.log(5e3) * 2.0 * np.arange(rot // 2) / rot).astype(np.float32))
    kp, vp = _pages(6, nkv, hd, dtype)
    table = _i32([[4, -1, -1], [-1, 5, 2]])   # sequence 1: base 1, so page index 2 is column 1 -> page 5
    base = _i32([0, 1])
    q_out = torch.empty(n, nh * hd, dtype=dtype, device=DEV)
    K.qk_norm_rope_kv(q.to(DEV), k.to(DEV), v.to(DEV), q_out, qg.to(DEV), kg.to(DEV), 1e-6, 2e-6, inv.to(DEV), 0.25,
                      _i32(tok_seq), _i32(tok_pos), kp, vp, table, base, nh, nkv, hd)
    pos = torch.tensor(tok_pos, dtype=torch.float64)
    ang = P.rope_angles(pos, rot, 5e3, 4.0)
    q_ref = P.apply_rope(P.rms_norm(q.double().view(n, nh, hd), qg.double(), 1e-6, add_one=False), ang)
    k_ref = P.apply_rope(P.rms_norm(k.double().view(n, nkv, hd), kg.double(), 2e-6, add_one=False), ang)
    tol = dict(atol=3e-6, rtol=3e-6) if dtype == torch.float32 else dict(atol=2e-2, rtol=1e-2)
    assert torch.allclose(q_out.cpu().double().view(n, nh, hd), q_ref, **tol)
    page_of = {0: {0: 4}, 1: {2: 5}}
    for t, (b, p) in enumerate(zip(tok_seq, tok_pos)):
        pg, row = page_of[b][p // 64], p % 64
        assert torch.allclose(kp[pg, :, row, :].cpu().double(), k_ref[t], **tol)
        assert torch.equal(vp[pg, :, :, row].cpu().view(-1), v[t])            # v is stored as it is
    # rows that no token wrote stay zero
    written = {(page_of[b][p // 64], p % 64) for b, p in zip(tok_seq, tok_pos)}
    mask = torch.ones(6, 64, dtype=torch.bool)
    for pg, row in written:
        mask[pg, row] = False
    assert float(kp.cpu().float().abs().sum(dim=(1, 3))[mask].sum()) == 0.0


@pytest.mark.parametrize("hd,nh,nkv,seqs,gains,rotates", [
    (256, 8, 4, [(0, 256)], True, True),                             # whole groups of four positions only
    (256, 8, 4, [(3, 130), (61, 71), (126, 66)], True, True),        # groups that begin and end inside of a wave's four tokens
    (256, 5, 3, [(62, 3), (1, 381)], False, True),
    (128, 16, 4, [(5, 1), (2, 2), (63, 190)], True, True),
    (128, 6, 1, [(1, 439)], True, False),
    (128, 16, 0, [(7, 193)], True, True),                            # a layer that reads another one's cache
    (256, 5, 3, [(62, 3), (1, 701)], False, True),                   # (above every line of the rule)
    (128, 16, 4, [(5, 1), (2, 2), (63, 301)], True, True),
    (128, 6, 1, [(1, 739)], True, False),
    (128, 16, 0, [(7, 493)], True, True),
])
def test_qk_norm_rope_kv_of_many_tokens(K, hd, nh, nkv, seqs, gains, rotates):
    """Steps of many tokens over pages in tile order, which take a kernel of their own: against 64-bit rows (bfloat16 rounds to
    2^-9 of a value; a rotated pair's two 32-bit products are far below that), values as they are, other rows untouched."""
    g = torch.Generator().manual_seed(hd + nh)
    tok_seq = [b for b, (_, m) in enumerate(seqs) for _ in range(m)]
    tok_pos = [p + i for p, m in seqs for i in range(m)]
    n, width = len(tok_pos), max((p + m + 63) // 64 for p, m in seqs)
    assert n * (nh + nkv) >= 3072
    qkv = torch.randn(n, (nh + 2 * nkv) * hd, generator=g).bfloat16()
    q, k, v = qkv[:, :nh * hd], qkv[:, nh * hd:(nh + nkv) * hd], qkv[:, (nh + nkv) * hd:]
    qg, kg = ((torch.randn(hd, generator=g) * 0.1 + 1) for _ in range(2)) if gains else (None, None)
    inv = torch.from_numpy(np.exp(-np.log(1e6) * 2.0 * np.arange(hd // 2) / hd).astype(np.float32)) if rotates else None
    pages = len(seqs) * width
    table = torch.randperm(pages, generator=g).to(torch.int32).view(len(seqs), width)
    kp = torch.zeros(pages, max(nkv, 1), 64, hd, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros(pages, max(nkv, 1), hd, 64, dtype=torch.bfloat16, device=DEV)
    dev = lambda x: x.to(DEV) if x is not None else None
    on = qkv.to(DEV)
    q_out = torch.empty(n, nh * hd, dtype=torch.bfloat16, device=DEV)
    keys = (on[:, nh * hd:(nh + nkv) * hd], on[:, (nh + nkv) * hd:]) if nkv else (None, None)
    K.qk_norm_rope_kv(on[:, :nh * hd], *keys, q_out, dev(qg), dev(kg), 1e-6, 2e-6, dev(inv), 0.125, _i32(tok_seq), _i32(tok_pos),
                      kp if nkv else None, vp if nkv else None, table.to(DEV), _i32([0] * len(seqs)), nh, nkv, hd, True)
    pos = torch.tensor(tok_pos, dtype=torch.float64)

    def want(x, gain, eps, heads):
        x = x.double().reshape(n, heads, hd)
        if gain is not None:
            x = P.rms_norm(x, gain.double(), eps, add_one=False)
        return P.apply_rope(x, P.rope_angles(pos, hd, 1e6, 8.0)) if rotates else x
    # (the kernel's angles are 32-bit products: at position 500 they are off by up to 3e-5)
    tol = dict(atol=2e-4, rtol=2 ** -8)
    assert torch.allclose(q_out.cpu().double().view(n, nh, hd), want(q, qg, 1e-6, nh), **tol)
    if not nkv:
        return
    # tile order, back to [page, kv head, 64, hd]: keys are tiles of 16 rows by 32 elements, values of 16 elements by 32 rows
    k_rows = kp.cpu().view(pages, nkv, 4, hd // 32, 4, 16, 8).permute(0, 1, 2, 5, 3, 4, 6).reshape(pages, nkv, 64, hd)
    v_rows = vp.cpu().view(pages, nkv, hd // 16, 2, 4, 16, 2, 4).permute(0, 1, 3, 6, 4, 7, 2, 5).reshape(pages, nkv, 64, hd)
    page = torch.tensor([int(table[b, p // 64]) for b, p in zip(tok_seq, tok_pos)])
    row = torch.tensor([p % 64 for p in tok_pos])
    assert torch.allclose(k_rows[page, :, row].double(), want(k, kg, 2e-6, nkv), **tol)
    assert torch.equal(v_rows[page, :, row], v.reshape(n, nkv, hd))
    written = torch.zeros(pages, 64, dtype=torch.bool)
    written[page, row] = True
    assert float(k_rows.float().abs().sum((1, 3))[~written].sum()) == 0 == float(v_rows.float().abs().sum((1, 3))[~written].sum())


@pytest.mark.parametrize("hd,nh,nkv", [(256, 8, 4), (256, 3, 9), (128, 5, 5), (128, 32, 16)])
@pytest.mark.parametrize("first", [512, 513, 514, 515])
def test_qk_norm_rope_kv_of_a_windows_pages(K, hd, nh, nkv, first):
    """A prompt's later piece on a layer with a window: the tables begin at a page of their own, a page is not there and one is no
    page of the pool.  Sequences of many tokens and of few, begun at every place of a group of four, ended at each, two tokens of
    one position after the other.  The kernel of many tokens against the one of few (a token's rows differ by the order of a
    sum and by the sine's last bits: half a unit of bfloat16's eight places each); values and untouched rows are the same."""
    g = torch.Generator().manual_seed(hd + nh + first)
    seqs = [(first, 389), (first + 91, 1), (130, 2), (131, 2), (133, 3), (first + 2, 5), (77, 6), (192, 7), (63, 2), (70, 601 - first % 7)]
    tok_seq = [b for b, (_, m) in enumerate(seqs) for _ in range(m)]
    tok_pos = [p + i for p, m in seqs for i in range(m)]
    n, base = len(tok_pos), [max(0, p // 64 - b % 2) for b, (p, _) in enumerate(seqs)]
    width = max((p + m - 1) // 64 + 1 - a for (p, m), a in zip(seqs, base))
    assert n * (nh + nkv) >= 9216 and n >= 8 * len(seqs)
    pages = len(seqs) * width
    table = torch.randperm(pages, generator=g).to(torch.int32).view(len(seqs), width)
    table[0, 3], table[9, 2] = -1, pages
    on = torch.randn(n, (nh + 2 * nkv) * hd, generator=g).bfloat16().to(DEV)
    q, k, v = on[:, :nh * hd], on[:, nh * hd:(nh + nkv) * hd], on[:, (nh + nkv) * hd:]
    gains = [(torch.randn(hd, generator=g) * 0.1 + 1).to(DEV) for _ in range(2)]
    inv = torch.exp(-torch.arange(hd // 2) * (26.0 / hd)).float().to(DEV)
    got = []
    for apart in (len(seqs), n):                    # (fewer than eight tokens a sequence: the kernel of few tokens)
        q_out = torch.empty(n, nh * hd, dtype=torch.bfloat16, device=DEV)
        kp, vp = torch.full((pages, nkv, 64, hd), 3.0, dtype=torch.bfloat16, device=DEV), torch.full((pages, nkv, hd, 64), 3.0, dtype=torch.bfloat16, device=DEV)
        K.qk_norm_rope_kv(q, k, v, q_out, *gains, 1e-6, 2e-6, inv, 0.125, _i32(tok_seq), _i32(tok_pos), kp, vp, table.to(DEV), _i32(base), nh, nkv, hd, True, apart)
        got.append((q_out.double(), kp.double(), vp))
    (q0, k0, v0), (q1, k1, v1) = got
    assert torch.equal(v0, v1) and torch.equal(k0 == 3.0, k1 == 3.0)
    near = lambda a, b: bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2e-4).all())
    assert near(q0, q1) and near(k0, k1) and float((q0 != q1).double().mean()) < 0.01 and float((k0 != k1).double().mean()) < 0.01
    there = torch.tensor([0 <= int(table[b, p // 64 - base[b]]) < pages for b, p in zip(tok_seq, tok_pos)], device=DEV)
    assert 0 < int(there.sum()) < n and int((v0 != 3.0).sum()) == int((v[there] != 3.0).sum())


@pytest.mark.parametrize("pos", [0, 1, 10, 100, 1000])
def test_rope_golden(K, pos):
    # research/kernels/generate_golden.py:140-155: nh 4, hd 256, theta 1e4, no norm
    q, want = _g(f"rope_nh4_hd256_pos{pos}_q_in"), _g(f"rope_nh4_hd256_pos{pos}_q_out")
    inv = torch.from_numpy(np.exp(-np.log(1e4) * 2.0 * np.arange(128) / 256).astype(np.float32))
    q_out = torch.empty(1, 1024, dtype=torch.float32, device=DEV)
    K.qk_norm_rope_kv(q.view(1, -1).to(DEV), None, None, q_out, None, None, 0.0, 0.0, inv.to(DEV), 1.0,
                      _i32([0]), _i32([pos]), None, None, None, None, 4, 0, 256)
    assert torch.allclose(q_out.cpu().view(-1), want, atol=3e-4 if pos >= 100 else 2e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_geglu(K, dtype):
    n, ff = 5, 333
    gu = (torch.randn(n, 2 * ff) * 2).to(dtype).to(DEV)
    out = torch.empty(n, ff, dtype=dtype, device=DEV)
    K.geglu(gu[:, :ff], gu[:, ff:], out)
    ref = P.gelu_tanh(gu[:, :ff].cpu().double()) * gu[:, ff:].cpu().double()
    assert torch.allclose(out.cpu().double(), ref, **_tol(dtype))
    big = torch.tensor([[-100.0, 100.0, 1.0, 1.0]], device=DEV)
    o = torch.empty(1, 2, device=DEV)
    K.geglu(big[:, :2], big[:, 2:], o)
    assert torch.isfinite(o).all() and float(o[0, 1]) == 100.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("activation", ["gelu_tanh", "silu", "gelu", "relu"])
def test_gated_act_takes_the_activation_as_a_parameter(K, dtype, activation):
    """out = act(gate) * up for every activation the kernel knows, against the library's functions
    in 64-bit; large arguments of either sign stay finite."""
    n, ff = 7, 301
    gu = (torch.randn(n, 2 * ff, generator=torch.Generator().manual_seed(5)) * 3).to(dtype)
    gu[0, :4] = torch.tensor([-90.0, 90.0, -30.0, 30.0]).to(dtype)
    out = torch.full((n, ff), float("nan"), dtype=dtype, device=DEV)
    K.gated_act(gu[:, :ff].to(DEV), gu[:, ff:].to(DEV), out, activation)
    g, u = gu[:, :ff].double(), gu[:, ff:].double()
    act = {"gelu_tanh": P.gelu_tanh, "silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu,
           "relu": torch.relu}[activation]
    assert torch.isfinite(out.float()).all()
    assert torch.allclose(out.cpu().double(), act(g) * u, **_tol(dtype))
    with pytest.raises(ValueError, match="unknown activation"):
        K.gated_act(gu[:, :ff].to(DEV), gu[:, ff:].to(DEV), out, "swish_of_tomorrow")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_add_bias_to_rows_of_a_wider_matrix(K, dtype):
    """y[r] += bias, summed in 32-bit and rounded once; the columns beside the rows' stretch stay."""
    n, cols = 9, 203
    g = torch.Generator().manual_seed(6)
    wide = torch.randn(n, cols + 13, generator=g).to(dtype).to(DEV)
    before = wide.clone()
    bias = torch.randn(cols, generator=g).to(DEV)
    K.add_bias(wide[:, 5:5 + cols], bias)
    want = (before[:, 5:5 + cols].float() + bias).to(dtype)
    assert torch.equal(wide[:, 5:5 + cols], want)
    assert torch.equal(wide[:, :5], before[:, :5]) and torch.equal(wide[:, 5 + cols:], before[:, 5 + cols:])
    with pytest.raises(TypeError):
        K.add_bias(wide[:, 5:5 + cols], bias[:-1])


@pytest.mark.parametrize("scale,cap", [(1.0, 30.0), (2.5, 4.0), (0.125, 0.0)])
def test_scale_and_soft_cap_of_logits(K, scale, cap):
    """x <- cap tanh(scale x / cap), or scale x without a cap; huge logits end at the cap, not at NaN."""
    x = torch.randn(5, 1001, generator=torch.Generator().manual_seed(7)) * 6
    x[0, :3] = torch.tensor([1e6, -1e6, 0.0])
    y = x.to(DEV)
    K.scale_cap(y, scale, cap)
    want = x.double() * scale
    if cap > 0:
        want = cap * torch.tanh(want / cap)
    assert torch.isfinite(y).all()
    assert torch.allclose(y.cpu().double(), want, atol=2e-6 * max(cap, 1.0), rtol=2e-6)
    with pytest.raises(ValueError):
        K.scale_cap(y, 1.0, -1.0)


@pytest.mark.parametrize("n", [128, 1152, 6912])
def test_gelu_golden(K, n):
    x, want = _g(f"gelu_n{n}_x"), _g(f"gelu_n{n}_out")
    out = torch.empty(1, n, device=DEV)
    K.geglu(x.view(1, n).to(DEV), torch.ones(1, n, device=DEV), out)
    assert torch.allclose(out.cpu().view(-1), want, atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("ta,tw,tc", [(torch.float32,) * 3, (torch.bfloat16,) * 3,
                                      (torch.bfloat16, torch.bfloat16, torch.float32),
                                      (torch.bfloat16, torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("m,n,k", [(1, 53, 29), (37, 130, 75), (65, 64, 16)])
def test_gemm_plain(K, ta, tw, tc, m, n, k):
    a, w = torch.randn(m, k).to(ta), torch.randn(n, k).to(tw)
    c = torch.empty(m, n, dtype=tc, device=DEV)
    K.gemm_plain(a.to(DEV), w.to(DEV), c)
    ref = a.double() @ w.double().T
    tol = dict(atol=1e-5, rtol=1e-5) if tc == torch.float32 else dict(atol=5e-2, rtol=1e-2)
    assert torch.allclose(c.cpu().double(), ref, **tol)
    # a strided input (a slice of a wider matrix)
    wide = torch.randn(m, k + 11).to(ta).to(DEV)
    K.gemm_plain(wide[:, 5:5 + k], w.to(DEV), c)
    assert torch.allclose(c.cpu().double(), wide[:, 5:5 + k].cpu().double() @ w.double().T, **tol)


@pytest.mark.parametrize("ta,tw", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 96, 300])
@pytest.mark.parametrize("n,k", [(1, 4), (16, 64), (17, 1028), (63, 36), (130, 515), (2100, 260)])
def test_gemm_plain_tiles(K, ta, tw, m, n, k):
    """Edges of the tiles of rows, columns and k, whole and broken stretches of four, and rows that are not aligned.
    Sums of K products in 32-bit are off by at most K 2^-24 of the sum of their sizes."""
    g = torch.Generator().manual_seed(m * 7 + n)
    a, w = torch.randn(m, k + 3, generator=g).to(ta).to(DEV), torch.randn(n, k, generator=g).to(tw).to(DEV)
    for x in (a[:, :k].contiguous(), a[:, 3:]):
        c = torch.full((m + 1, n + 2), 7.0, device=DEV)
        K.gemm_plain(x, w, c[:m, :n])
        bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert bool(((c[:m, :n].double() - x.double() @ w.double().T).abs() <= bound).all())
        assert bool((c[m] == 7.0).all()) and bool((c[:, n:] == 7.0).all())       # nothing outside is written


@pytest.mark.parametrize("ta,tw", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16),
                                   (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("m,n,k", [(257, 3300, 36), (300, 3300, 515), (320, 4161, 260), (1100, 960, 129),           # tiles of 64 rows
                                   (97, 5500, 68), (200, 2400, 131),                                                 # of 32
                                   (17, 16400, 257), (64, 8200, 259), (33, 8200, 515),                               # of 32 for few rows that fours do not fit
                                   (2, 70, 33), (2, 515, 1027), (1, 33, 4097)])                                      # a wave a column
def test_gemm_plain_large_tiles_and_odd_rows(K, ta, tw, m, n, k):
    """Enough tiles to fill the chip, their last rows and columns broken, whole and broken stretches of k; and rows that four
    elements do not fit, few and many.  Every output is within K 2^-24 of the sum of its products' sizes."""
    g = torch.Generator().manual_seed(m * 7 + n)
    a, w = torch.randn(m, k + 3, generator=g).to(ta).to(DEV), torch.randn(n, k, generator=g).to(tw).to(DEV)
    for x in (a[:, :k].contiguous(), a[:, 3:]):
        c = torch.full((m + 1, n + 2), 7.0, device=DEV)
        K.gemm_plain(x, w, c[:m, :n])
        bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert bool(((c[:m, :n].double() - x.double() @ w.double().T).abs() <= bound).all())
        assert bool((c[m] == 7.0).all()) and bool((c[:, n:] == 7.0).all())


# Up to eight rows whose fours fit: workgroups of 16, 8 and 4 waves (256 and 512 blocks of eight columns are the lines between them), a
# broken last block, chunks of 64 columns that break off, one chunk in all, and as many chunks a wave as are in flight, more or less.
@pytest.mark.parametrize("ta,tw", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("n", [7, 2048, 2050, 4096, 4101, 9001])
@pytest.mark.parametrize("k", [4, 60, 64, 68, 256, 772, 1028, 2052, 3084, 4164])
def test_gemm_plain_up_to_eight_rows(K, ta, tw, n, k):
    g = torch.Generator().manual_seed(n + k)
    w = torch.randn(n, k, generator=g).to(tw).to(DEV)
    for m in (1, 3, 8):
        x = torch.randn(m, k + 4, generator=g).to(ta).to(DEV)[:, :k]
        c = torch.full((m + 1, n + 2), 7.0, device=DEV)
        K.gemm_plain(x, w, c[:m, :n])
        bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert bool(((c[:m, :n].double() - x.double() @ w.double().T).abs() <= bound).all())
        assert bool((c[m] == 7.0).all()) and bool((c[:, n:] == 7.0).all())
    x[1, k - 1], x[2, 0], w[5, 2] = float("nan"), float("inf"), float("-inf")          # they stay in their rows and columns
    K.gemm_plain(x, w, c[:m, :n])
    got, plain = c[:m, :n].cpu(), torch.ones(m, n, dtype=torch.bool)
    plain[1], plain[2], plain[:, 5] = False, False, False
    assert bool(got[1].isnan().all()) and bool(got[plain].isfinite().all())
    assert not bool(got[2, :5].isfinite().any()) and not bool(got[0, 5].isfinite())


@pytest.mark.parametrize("ff,k", [(2049, 516), (3080, 512), (3073, 4), (5376, 2048), (2056, 772)])
@pytest.mark.parametrize("activation", ["gelu_tanh", "silu", "swish_clamped"])
def test_gemm_gated_few_rows(K, ff, k, activation):
    """Gate and up of up to eight rows with their activation in one kernel, against the product and the activation in a row (their
    sums begin at another chunk of columns for another block, so they differ by rounding: either is within k 2^-24 of its
    products' sizes, which the forms here pass on at most 1.2-fold): a broken last block of columns, rows that lie apart; what
    it does not take is refused."""
    g = torch.Generator(device=DEV).manual_seed(ff + k)
    w = torch.randn(2 * ff, k, device=DEV, generator=g) * k ** -0.5
    for m in (1, 3, 8):
        x = torch.randn(m, k + 4, device=DEV, generator=g)[:, :k]
        out, gu, want = torch.full((m + 1, ff + 2), 7.0, device=DEV), torch.empty(m, 2 * ff, device=DEV), torch.empty(m, ff, device=DEV)
        assert K.gemm_gated(x, w, out[:m, :ff], activation, 1.5, 0.7)
        K.gemm_plain(x, w, gu)
        K.gated_act(gu[:, :ff], gu[:, ff:], want, activation, 1.5, 0.7)
        size = x.abs() @ w.abs().T
        off = 1.2 * 2 * k * 2.0 ** -24 * (size[:, :ff] * (gu[:, ff:].abs() + 1.0) + size[:, ff:] * gu[:, :ff].abs()) + 1e-6 * want.abs()
        assert bool(((out[:m, :ff] - want).abs() <= off).all()) and float((out[:m, :ff] - want).norm()) <= 1e-6 * float(want.norm())
        assert bool((out[m] == 7.0).all()) and bool((out[:, ff:] == 7.0).all())
    x = torch.randn(9, k + 4, device=DEV, generator=g)
    out = torch.empty(9, ff, device=DEV)
    assert not K.gemm_gated(x[:, :k], w, out) and not K.gemm_gated(x[:3, 1:k + 1], w, out[:3])
    assert not K.gemm_gated(x[:3, :k].bfloat16(), w, out[:3]) and not K.gemm_gated(x[:3, :k].contiguous(), w[:2048], out[:3, :1024])


def test_gemm_plain_up_to_eight_rows_rounds_alike(K):
    """Sums are no longer on one side of the lines between the kernels than on the other: 16 waves share K up to 2,048 columns, 8 up to
    4,096 (the same products a sum, so the same error but for chance, some 1 % over 16,000 results) and 4 beyond (twice as
    many, and rounding grows as the root)."""
    g = torch.Generator().manual_seed(3)
    k, err = 5376, {}
    for n in (2048, 2304, 5376):
        x, w = torch.randn(8, k, generator=g).to(DEV), torch.randn(n, k, generator=g).to(DEV)
        for m in (3, 8):
            c = torch.empty(m, n, device=DEV)
            K.gemm_plain(x[:m], w, c)
            ref = x[:m].double() @ w.double().T
            err[m, n] = float((c.double() - ref).pow(2).mean().sqrt() / ref.pow(2).mean().sqrt())
    for m in (3, 8):
        assert err[m, 2304] <= 1.06 * err[m, 2048], err
        assert err[m, 5376] <= math.sqrt(2) * err[m, 2048], err


# Tiles whose stages of 32 columns come by themselves: 32 x 128 (also for up to 64 rows) and 128 x 128,
# their last rows and columns broken, one stage, two, three and more, whole and broken.
@pytest.mark.parametrize("m,n", [(33, 8200), (64, 8250), (17, 16400), (32, 16390),
                                 (300, 4000), (70, 10700), (65, 8190), (777, 10700), (257, 10700), (300, 10752)])
@pytest.mark.parametrize("k", [4, 28, 32, 36, 64, 92, 100, 132, 516])
def test_gemm_plain_rings(K, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k + 8, generator=g).to(DEV), torch.randn(n, k + 4, generator=g).to(DEV)[:, :k]
    x = a[:, 4:4 + k]
    c = torch.full((m + 1, n + 2), 7.0, device=DEV)
    K.gemm_plain(x, w, c[:m, :n])
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((c[:m, :n].double() - x.double() @ w.double().T).abs() <= bound).all())
    assert bool((c[m] == 7.0).all()) and bool((c[:, n:] == 7.0).all())
    x[1, k - 1], x[m - 1, 0], w[5, 2], w[n - 1, k - 2] = float("nan"), float("inf"), float("-inf"), float("inf")
    K.gemm_plain(x, w, c[:m, :n])                                  # they stay in their rows and columns
    plain = torch.ones(m, n, dtype=torch.bool, device=DEV)
    plain[[1, m - 1]] = False
    plain[:, [5, n - 1]] = False
    assert bool(c[1, :n].isnan().all()) and bool(c[:m, :n][plain].isfinite().all())
    assert not bool(c[:m, :n][~plain].isfinite().any())


@pytest.mark.parametrize("m,n,k", [(2, 40, 17), (70, 40, 18), (300, 3300, 20), (290, 3300, 18), (97, 5500, 20), (17, 16400, 258), (40, 8200, 257)])
def test_gemm_plain_special_values_in_every_kernel(K, m, n, k):
    """A NaN or an infinity stays in its row and column, and zeros behind the last k meet zeros only."""
    a, w = torch.ones(m, k, device=DEV), torch.ones(n, k, device=DEV)
    a[1, k - 1], w[5, 2] = float("nan"), float("inf")
    c = torch.empty(m, n, device=DEV)
    K.gemm_plain(a, w, c)
    want = torch.full((m, n), float(k), device=DEV)
    want[:, 5] = float("inf")
    want[1] = float("nan")
    assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c[~c.isnan()], want[~want.isnan()])


def test_gemm_plain_special_values(K):
    """A NaN or an infinity stays in its row and column, and zeros behind the last k meet zeros only."""
    for m in (3, 70):
        a, w = torch.ones(m, 18, device=DEV), torch.ones(40, 18, device=DEV)
        a[1, 17], w[5, 2] = float("nan"), float("inf")
        c = torch.empty(m, 40, device=DEV)
        K.gemm_plain(a, w, c)
        want = torch.full((m, 40), 18.0, device=DEV)
        want[:, 5] = float("inf")
        want[1] = float("nan")
        assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c[~c.isnan()], want[~want.isnan()])


def _attn_case(K, dtype, nh, nkv, hd, lens, window, scale, seed=0, boost=None):
    """Sequences of the given lengths in scattered pages; every position is a query."""
    g = torch.Generator().manual_seed(seed)
    n_pages = sum((L + 63) // 64 for L in lens) + 3
    kp, vp = _pages(n_pages, nkv, hd, dtype)
    perm = torch.randperm(n_pages, generator=g).tolist()
    width = max((L + 63) // 64 for L in lens)
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    ks, vs, qs, tok_seq, tok_pos = [], [], [], [], []
    for b, L in enumerate(lens):
        k = torch.randn(L, nkv, hd, generator=g).to(dtype)
        v = torch.randn(L, nkv, hd, generator=g).to(dtype)
        q = torch.randn(L, nh, hd, generator=g).to(dtype)
        if boost is not None:                  # one far key must win for the last query:
            k = k - k.mean(dim=-1, keepdim=True)   # every other key is orthogonal to that query (score 0),
            k[boost] = 1.0                         # the far key scores 20
            q[L - 1] = 20.0 / (hd * scale)
        for i in range((L + 63) // 64):
            pg = perm.pop()
            table[b, i] = pg
            rows = slice(i * 64, min(L, i * 64 + 64))
            kp[pg, :, :rows.stop - rows.start, :] = k[rows].transpose(0, 1).to(DEV)
            vp[pg, :, :, :rows.stop - rows.start] = v[rows].permute(1, 2, 0).to(DEV)
        ks.append(k); vs.append(v); qs.append(q)
        tok_seq += [b] * L
        tok_pos += list(range(L))
    q_all = torch.cat(qs).reshape(-1, nh * hd).to(DEV)
    out = torch.empty_like(q_all)
    K.attn_plain(q_all, out, kp, vp, table.to(DEV), _i32([0] * len(lens)), _i32(tok_seq), _i32(tok_pos),
                 nh, nkv, hd, scale, window)
    refs = [P.attention_core(q.double(), k.double(), v.double(), scale, window) for q, k, v in zip(qs, ks, vs)]
    return out.cpu().double().view(-1, nh, hd), torch.cat(refs), vs


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 40, None), (6, 1, 16, 70), (5, 5, 72, 300), (2, 1, 256, 64)])
def test_attn_plain(K, dtype, nh, nkv, hd, window):
    got, ref, _ = _attn_case(K, dtype, nh, nkv, hd, [1, 77, 300, 64], window, 0.21)
    # 32-bit: a score is a sum of hd products of N(0,1) values, so its rounding error, and with it
    # the relative error of exp(score), grows with hd
    tol = dict(atol=2e-6 + 1e-7 * hd, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    assert torch.allclose(got, ref, **tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,window", [(16, 4, 128, None), (20, 1, 6, 70), (32, 2, 34, None), (3, 1, 512, 130), (1, 1, 2, 1), (17, 1, 130, None)])
def test_attn_plain_rows(K, dtype, nh, nkv, hd, window):
    """Rows of several heads and tokens a workgroup: sequences that change within one, more heads on a key head than it takes,
    head sizes at the edges of its tiles and not a multiple of four; and one token a sequence, alone and with several
    workgroups to a row's pages."""
    from agave_amd.parts import Workspace
    lens = [1, 2, 1, 5, 130, 64, 65, 1, 300]
    scale = hd ** -0.5
    got, ref, _ = _attn_case(K, dtype, nh, nkv, hd, lens, window, scale)
    tol = dict(atol=2e-6 + 1e-7 * hd, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    assert torch.allclose(got, ref, **tol)
    real, asked = K.attn_plain, {}

    def last_tokens(q, out, kp, vp, table, base, tok_seq, tok_pos, *rest):
        """The same call for every sequence's last token."""
        ends = torch.tensor([sum(lens[:i + 1]) - 1 for i in range(len(lens))], device=DEV)
        for name, more in (("alone", {}), ("shared", {"span": 5, "workspace": Workspace(torch.device(DEV))})):
            o = torch.empty(len(lens), nh * hd, dtype=q.dtype, device=DEV)
            real(q[ends].contiguous(), o, kp, vp, table, base, tok_seq[ends].contiguous(), tok_pos[ends].contiguous(), *rest,
                 one_token_each=True, **more)
            asked[name] = o.cpu().double().view(-1, nh, hd)
        real(q, out, kp, vp, table, base, tok_seq, tok_pos, *rest)
    K.attn_plain = last_tokens
    try:
        _, ref, _ = _attn_case(K, dtype, nh, nkv, hd, lens, window, scale)
    finally:
        K.attn_plain = real
    ends = [sum(lens[:i + 1]) - 1 for i in range(len(lens))]
    for o in asked.values():
        assert torch.allclose(o, ref[ends], **tol)


@pytest.mark.parametrize("hd", [32, 300])
@pytest.mark.parametrize("n", [90, 170])
def test_attn_plain_values_that_are_not_finite(K, n, hd):
    """What lies behind a token's position reaches no result, also where a later token of the same workgroup sees it (170 tokens
    go eight to a workgroup, and position 70 is the seventh of its eight; 90 go one by one); heads whose values are read
    ahead and with their products."""
    nh, nkv = 4, 2
    kp, vp = _pages(3, nkv, hd, torch.float32)
    kp.normal_()
    vp.normal_()
    q, out = torch.randn(n, nh * hd, device=DEV), torch.empty(n, nh * hd, device=DEV)
    args = (_i32([[0, 1, 2]]), _i32([0]), _i32([0] * n), _i32(list(range(n))), nh, nkv, hd, 0.2, None)
    K.attn_plain(q, out, kp, vp, *args)
    want = out.clone()
    vp[1, 0, 3, 6] = float("inf")                                        # position 70, element 3 of key head 0
    last = n // 64
    vp[last, :, :, n % 64:] = float("nan")                                # positions that no token has
    kp[last, :, n % 64:] = float("nan")
    K.attn_plain(q, out, kp, vp, *args)
    bad = ~torch.isfinite(out)
    hit = torch.zeros(n, nh, hd, dtype=torch.bool, device=DEV)
    hit[70:, :2, 3] = True
    assert torch.equal(bad.view(n, nh, hd), hit)
    assert torch.allclose(out[~bad], want[~bad], atol=1e-6 * (1 + hd / 100), rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("spoil", ["query", "page", "key of no weight", "value"])
def test_attn_plain_rows_that_are_not_a_number(K, dtype, spoil):
    """A token whose query, or a key or value that it sees, is not a number: its heads' results say so, with one workgroup to a
    row and with several, also where a share of its pages has no other score or no weight; all other rows stay as they are."""
    from agave_amd.parts import Workspace
    nh, nkv, hd, B, ctx = 4, 2, 40, 2, 330
    g = torch.Generator().manual_seed(5)
    kp, vp = (torch.randn(6 * B, nkv, *shape, generator=g).to(dtype).to(DEV) for shape in ((64, hd), (hd, 64)))
    q = torch.randn(B, nh * hd, generator=g).to(dtype).to(DEV)
    table = torch.arange(6 * B, dtype=torch.int32, device=DEV).view(B, 6)
    hit = torch.zeros(B, nh, hd, dtype=torch.bool, device=DEV)

    def both():
        outs = []
        for more in ({}, {"span": 6, "workspace": Workspace(torch.device(DEV))}):
            out = torch.empty_like(q)
            K.attn_plain(q, out, kp, vp, table, _i32([0] * B), _i32(list(range(B))), _i32([ctx - 1] * B), nh, nkv, hd, 0.2, None,
                         one_token_each=True, **more)
            outs.append(out.view(B, nh, hd))
        return outs
    if spoil == "key of no weight":           # (page 4's scores exceed all others by some 300: nothing else has a weight)
        kp[4, 0] = 0.0
        kp[4, 0, :, 0] = 300.0 / 0.2
        q.view(B, nh, hd)[0, :2, 0] = 1.0
    want = both()
    if spoil == "query":
        q.view(B, nh, hd)[0, 1] = float("nan")
        hit[0, 1] = True
    elif spoil == "page":                     # (every score of one share)
        kp[2, 0] = float("nan")
        hit[0, :2] = True
    elif spoil == "key of no weight":
        kp[1, 0, 7] = float("nan")
        hit[0, :2] = True
    else:
        vp[1, 1, 3, 7] = float("nan")
        hit[0, 2:, 3] = True
    for got, ref in zip(both(), want):
        assert torch.equal(got.isnan(), hit)
        # (values that are not finite are summed element by element, in another order than the matrix cores')
        tol = dict(atol=1e-6, rtol=1e-5) if dtype == torch.float32 else dict(atol=1e-2, rtol=1e-2)
        assert torch.allclose(got[~hit], ref[~hit], **tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd,k_at,v_at", [(40, 0, 1), (40, 0, 4), (40, 1, 0), (34, 0, 2), (300, 3, 3)])
def test_attn_plain_pages_at_any_element(K, dtype, hd, k_at, v_at):
    """Pages that begin at any element of a buffer give the results of aligned ones, in prompts and decode steps."""
    from agave_amd.parts import Workspace
    nh, nkv, n = 4, 2, 150
    g = torch.Generator().manual_seed(hd + k_at)
    kp, vp = (torch.randn(3, nkv, *shape, generator=g).to(dtype).to(DEV) for shape in ((64, hd), (hd, 64)))
    q = torch.randn(n, nh * hd, generator=g).to(dtype).to(DEV)

    def moved(x, at):
        return torch.zeros(x.numel() + at, dtype=dtype, device=DEV)[at:].view(x.shape).copy_(x)
    table = _i32([[0, 1, 2]])
    outs = []
    for k, v in ((kp, vp), (moved(kp, k_at), moved(vp, v_at))):
        out = torch.empty_like(q)
        K.attn_plain(q, out, k, v, table, _i32([0]), _i32([0] * n), _i32(list(range(n))), nh, nkv, hd, 0.2, None)
        last = torch.empty_like(q[-1:])
        K.attn_plain(q[-1:], last, k, v, table, _i32([0]), _i32([0]), _i32([n - 1]), nh, nkv, hd, 0.2, None, one_token_each=True,
                     span=3, workspace=Workspace(torch.device(DEV)))
        outs.append(torch.cat([out, last]))
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd", [(4, 4, 32), (6, 2, 40), (8, 2, 300)])
def test_attn_plain_steps_of_many_sequences(K, dtype, nh, nkv, hd):
    """Tokens of several sequences among those that a workgroup would take, in any order: each has the result it has alone,
    whether the sequences get a workgroup each, share a few, or go one after another in one."""
    g = torch.Generator().manual_seed(hd)
    seqs, ctx = 5, 150
    kp, vp = (torch.randn(3 * seqs, nkv, *shape, generator=g).to(dtype).to(DEV) for shape in ((64, hd), (hd, 64)))
    table = torch.randperm(3 * seqs, generator=g).view(seqs, 3).int().to(DEV)
    tok_seq = [0] * 90 + [1, 2, 3, 4, 0, 2] + [3] * 20 + torch.randint(0, seqs, (200,), generator=g).tolist()
    tok_pos = torch.randint(0, ctx, (len(tok_seq),), generator=g).tolist()
    n = len(tok_seq)
    q = torch.randn(n, nh * hd, generator=g).to(dtype).to(DEV)

    def go(rows, **more):
        out = torch.empty(len(rows), nh * hd, dtype=dtype, device=DEV)
        K.attn_plain(q[rows].contiguous(), out, kp, vp, table, _i32([0] * seqs), _i32([tok_seq[r] for r in rows]), _i32([tok_pos[r] for r in rows]),
                     nh, nkv, hd, 0.2, 70, **more)
        return out
    rows = list(range(n))
    want = go(rows, one_token_each=True)
    for most in (lambda run: 1, lambda run: 3, lambda run: run, None):
        assert torch.equal(go(rows, most_seqs=most), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 40, None), (3, 1, 512, 9), (5, 5, 2, None), (6, 2, 130, 20), (2, 2, 256, 70)])
@pytest.mark.parametrize("most_keys", [5, 16, 64])
def test_attn_plain_few_keys(K, dtype, nh, nkv, hd, window, most_keys):
    """Steps of few keys and rows, against the plain implementation; a sequence that sees more keys than it was said to is right
    all the same, also where what it does not see is not a number."""
    lens = [1, 2, min(most_keys, 40), 90 if most_keys == 64 else 70]
    real, rows = K.attn_plain, {}

    def few(q, out, kp, vp, table, base, tok_seq, tok_pos, *rest):
        n = 256 // nh                                             # (few rows: the first ones, and the last ones)
        for at in (slice(0, n), slice(q.shape[0] - n if q.shape[0] > n else 0, q.shape[0])):
            for junk in (False, True):
                if junk:
                    for b, L in enumerate(lens):
                        page = int(table[b, (L - 1) // 64])
                        if L % 64:
                            kp[page, :, L % 64:] = float("nan")
                            vp[page, :, :, L % 64:] = float("nan")
                o = torch.empty_like(q[at])
                real(q[at].contiguous(), o, kp, vp, table, base, tok_seq[at].contiguous(), tok_pos[at].contiguous(), *rest, most_keys=most_keys)
                rows[at.start, junk] = (at, o.cpu().double().view(-1, nh, hd))
        real(q, out, kp, vp, table, base, tok_seq, tok_pos, *rest)
    K.attn_plain = few
    try:
        _, ref, _ = _attn_case(K, dtype, nh, nkv, hd, lens, window, hd ** -0.5)
    finally:
        K.attn_plain = real
    tol = dict(atol=2e-6 + 1e-7 * hd, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    for at, got in rows.values():
        assert torch.allclose(got, ref[at], **tol)


@pytest.mark.parametrize("what", ["query", "key", "value"])
def test_attn_plain_few_keys_that_are_not_finite(K, what):
    """A NaN reaches the rows that see it, all of a head's elements or a value's own, and nothing else."""
    nh, nkv, hd, n = 4, 2, 24, 30
    g = torch.Generator().manual_seed(1)
    kp, vp = (torch.randn(1, nkv, *shape, generator=g).to(DEV) for shape in ((64, hd), (hd, 64)))
    q = torch.randn(n, nh * hd, generator=g).to(DEV)
    args = (_i32([[0]]), _i32([0]), _i32([0] * n), _i32(list(range(n))), nh, nkv, hd, 0.2, None)
    want, out = torch.empty_like(q), torch.empty_like(q)
    K.attn_plain(q, want, kp, vp, *args, most_keys=n)
    hit = torch.zeros(n, nh, hd, dtype=torch.bool, device=DEV)
    if what == "query":
        q.view(n, nh, hd)[7, 1, 3] = float("nan")
        hit[7, 1] = True
    elif what == "key":
        kp[0, 1, 17, 5] = float("nan")
        hit[17:, 2:] = True
    else:
        vp[0, 0, 9, 17] = float("inf")
        hit[17:, :2, 9] = True
    K.attn_plain(q, out, kp, vp, *args, most_keys=n)
    assert torch.equal(~torch.isfinite(out.view(n, nh, hd)), hit)
    assert torch.equal(out.view(n, nh, hd)[~hit], want.view(n, nh, hd)[~hit])


def test_attn_plain_far_key_wins(K):
    # among 700 keys, key 3 is made to dominate the last query's softmax: the output must be its value
    got, ref, vs = _attn_case(K, torch.float32, 2, 1, 32, [700], None, 0.5, seed=1, boost=3)
    assert torch.allclose(got[-1], ref[-1], atol=1e-5)
    assert torch.allclose(got[-1, 0], vs[0][3, 0].double(), atol=1e-2)
    # with a window that ends before it, the same key must not be seen
    got_w, ref_w, _ = _attn_case(K, torch.float32, 2, 1, 32, [700], 696, 0.5, seed=1, boost=3)
    assert torch.allclose(got_w[-1], ref_w[-1], atol=1e-5)
    assert not torch.allclose(got_w[-1, 0], vs[0][3, 0].double(), atol=1e-1)
    got_e, ref_e, _ = _attn_case(K, torch.float32, 2, 1, 32, [700], 697, 0.5, seed=1, boost=3)   # edge: just inside
    assert torch.allclose(got_e[-1, 0], vs[0][3, 0].double(), atol=1e-2)


@pytest.mark.parametrize("tag,nh,nkv,hd,sl,suffix", [
    ("sdpa_nh4_nkv1_hd256_sl256", 4, 1, 256, 256, "_naive"), ("sdpa_nh4_nkv1_hd256_sl64", 4, 1, 256, 64, "_online"),
    ("sdpa_nh20_nkv5_hd128_sl32", 20, 5, 128, 32, ""), ("sdpa_nh4_nkv1_hd256_sl1", 4, 1, 256, 1, "_naive")])
def test_attn_plain_golden(K, tag, nh, nkv, hd, sl, suffix):
    # research/kernels/generate_golden.py:56-95; the reference's criterion is max error < 1e-3
    # (tests/sdpa_harness.zig:124-136); 32-bit sums give far less
    q, keys, values = _g(tag + "_q"), _g(tag + "_keys").view(sl, nkv, hd), _g(tag + "_values").view(sl, nkv, hd)
    n_pages = (sl + 63) // 64
    kp, vp = _pages(n_pages, nkv, hd, torch.float32)
    for i in range(n_pages):
        rows = slice(i * 64, min(sl, i * 64 + 64))
        kp[i, :, :rows.stop - rows.start] = keys[rows].transpose(0, 1).to(DEV)
        vp[i, :, :, :rows.stop - rows.start] = values[rows].permute(1, 2, 0).to(DEV)
    out = torch.empty(1, nh * hd, device=DEV)
    K.attn_plain(q.view(1, -1).to(DEV), out, kp, vp, _i32([list(range(n_pages))]), _i32([0]), _i32([0]), _i32([sl - 1]),
                 nh, nkv, hd, 1.0 / math.sqrt(hd), None)
    assert torch.allclose(out.cpu().view(-1), _g(tag + "_out" + suffix), atol=2e-5)


# ---------------------------------------------------------------- sampling
@pytest.fixture(scope="module")
def S():
    from agave_amd.ops import sampling
    return sampling


def _sample(S, logits, params):
    lg = logits.to(DEV).float().contiguous()
    work = torch.empty_like(lg)
    out = torch.empty(lg.shape[0], dtype=torch.int32, device=DEV)
    S.sample(lg, work, torch.tensor(params, dtype=torch.float32, device=DEV), out)
    got = out.cpu().tolist()
    # with scratch, rows of a large vocabulary are shared among workgroups; what it held before must not matter
    class Row:
        def __init__(self, p):
            self.temperature, self.top_k, self.top_p = p[0], int(p[1]), p[2]
    for kinds in (S.KIND_ALL, S.kinds_of([Row(p) for p in params], lg.shape[1])):
        scratch = torch.randint(-2 ** 31, 2 ** 31 - 1, (S.scratch_words() * lg.shape[0],), dtype=torch.int32,
                                device=DEV).view(torch.float32)
        out.fill_(-1)
        S.sample(lg, work, torch.tensor(params, dtype=torch.float32, device=DEV), out, scratch, kinds=kinds)
        assert out.cpu().tolist() == got
    return got


def test_argmax_first_of_ties(S):
    lg = torch.full((3, 5000), -1.0)
    lg[0, [4000, 77, 3000]] = 2.0
    lg[1, :] = float("-inf")
    lg[2, 4999] = 0.5
    assert _sample(S, lg, [[0, 0, 1, 0.9]] * 3) == [77, 0, 4999]


@pytest.mark.parametrize("temperature,top_k,top_p", [(1.0, 0, 1.0), (0.7, 0, 1.0), (1.3, 5, 1.0), (1.0, 0, 0.6),
                                                      (0.9, 50, 0.8), (1.0, 2000, 0.95), (2.0, 1, 1.0)])
@pytest.mark.parametrize("vocab", [3001, 40013, 262208])
def test_sample_matches_plain_rule(S, temperature, top_k, top_p, vocab):
    """For every token the plain rule can draw, a u in the middle of its interval of the running
    sum must give exactly that token."""
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(vocab, generator=g) * 2.5
    w = P.sample_distribution(logits, temperature, top_k, top_p)
    cdf = torch.cumsum(w, 0) / w.sum()
    support = torch.nonzero(w > 0).view(-1).tolist()
    if top_k:
        assert len(support) <= min(top_k, 1024)
    picks = support if len(support) <= 64 else [support[i] for i in range(0, len(support), len(support) // 64)]
    us, want = [], []
    for i in picks:
        lo = float(cdf[i - 1]) if i > 0 else 0.0
        hi = float(cdf[i])
        if hi - lo < 1e-5:
            continue
        us.append((lo + hi) / 2)
        want.append(i)
    got = _sample(S, logits.view(1, -1).repeat(len(us), 1), [[temperature, top_k, top_p, u] for u in us])
    assert got == want
    assert all(P.sample_token(logits, temperature, top_k, top_p, u) == i for u, i in zip(us, want))


def test_sample_rows_are_independent_and_mixed(S):
    g = torch.Generator().manual_seed(6)
    lg = torch.randn(4, 70001, generator=g)
    params = [[0.0, 0, 1.0, 0.3], [0.8, 0, 1.0, 0.3], [0.8, 3, 1.0, 0.99], [1.0, 0, 0.5, 0.0]]
    together = _sample(S, lg, params)
    alone = [_sample(S, lg[i:i + 1], [params[i]])[0] for i in range(4)]
    assert together == alone
    assert together[0] == int(lg[0].argmax())
    assert together[2] in torch.topk(lg[2], 3).indices.tolist()
    assert together == [P.sample_token(lg[i], *params[i]) for i in range(4)]


@pytest.mark.parametrize("vocab", [3001, 4096, 40013])
@pytest.mark.parametrize("temperature,top_k,top_p", [(0.8, 0, 0.01), (1.7, 5000, 0.01), (1.0, 1000, 1.0),
                                                      (0.8, 0, 0.9), (1.3, 1024, 0.7), (1.0, 900, 0.5)])
def test_sample_with_more_equal_logits_than_the_filter_collects(S, vocab, temperature, top_k, top_p):
    """Some hundred logits above a plateau of far more than a thousand equal ones: the 1024 largest
    end inside the plateau, all of which stays or goes together, and the draw has to range over
    entries that the filter could not collect.  top_p = 0.01 keeps the maximum alone: its weight,
    which is exactly 1, has to equal the threshold wherever it is computed again."""
    g = torch.Generator().manual_seed(vocab + top_k)
    logits = torch.randn(vocab, generator=g) * 2.0
    plateau = float(torch.sort(logits, descending=True).values[700])
    logits[::3] = plateau                                  # vocab / 3 equal entries below about 470 others
    w = P.sample_distribution(logits, temperature, top_k, top_p)
    cdf = torch.cumsum(w, 0) / w.sum()
    support = torch.nonzero(w > 0).view(-1).tolist()
    picks = support if len(support) <= 48 else [support[i] for i in range(0, len(support), len(support) // 48)]
    picks = sorted(set(picks + support[-2:]))
    us, want = [], []
    for i in picks:
        lo = float(cdf[i - 1]) if i > 0 else 0.0
        hi = float(cdf[i])
        if hi - lo < 1e-5:
            continue
        us.append((lo + hi) / 2)
        want.append(i)
    assert us
    got = _sample(S, logits.view(1, -1).repeat(len(us), 1), [[temperature, top_k, top_p, u] for u in us])
    assert got == want


def test_sample_random_parameters_ties_and_masked_halves(S):
    """A sweep of random rows and parameters, some rows with a seventh of their entries equal and
    some with their upper half at -inf, six rows a batch with mixed kinds; every draw must be the
    plain rule's (a u within 1e-4 of an interval's edge may go to the neighbour)."""
    rng = np.random.default_rng(0)
    checked = 0
    for trial in range(48):
        vocab = int(rng.choice([4096, 5003, 40013]))
        g = torch.Generator().manual_seed(trial)
        lg = torch.randn(6, vocab, generator=g) * float(rng.choice([0.5, 2.0, 6.0]))
        if trial % 3 == 0:
            lg[:, ::7] = lg[:, 3:4]
        if trial % 4 == 0:
            lg[:, vocab // 2:] = float("-inf")
        params = [[float(rng.choice([0.0, 0.3, 0.8, 1.0, 1.7])), int(rng.choice([0, 0, 1, 5, 40, 1000, 1024, 5000])),
                   float(rng.choice([1.0, 1.0, 0.95, 0.7, 0.3, 0.01])), float(rng.random())] for _ in range(6)]
        got = _sample(S, lg, params)
        for b, (t, k, p, u) in enumerate(params):
            want = P.sample_token(lg[b], t, k, p, u)
            if got[b] != want:
                w = P.sample_distribution(lg[b], t, k, p)
                assert t > 0 and float(w[got[b]]) > 0, (trial, b, params[b], got[b], want)
                cdf = torch.cumsum(w, 0) / w.sum()
                edges = [float(cdf[got[b]])] + ([float(cdf[got[b] - 1])] if got[b] else [])
                assert min(abs(e - u) for e in edges) < 1e-4, (trial, b, params[b], got[b], want)
            checked += 1
    assert checked == 48 * 6


def test_sample_frequencies_follow_softmax(S):
    lg = torch.tensor([[0.0, 1.0, 2.0, -1.0, 0.5]])
    n = 4000
    us = (torch.arange(n) + 0.5) / n                    # a stratified sweep of u
    got = _sample(S, lg.repeat(n, 1), [[0.7, 0, 1.0, float(u)] for u in us])
    freq = torch.bincount(torch.tensor(got), minlength=5).double() / n
    assert torch.allclose(freq, torch.softmax(lg[0].double() / 0.7, 0), atol=2.0 / n)


def test_repeat_penalty(S):
    lg = torch.tensor([[2.0, -2.0, 1.0, 3.0], [2.0, -2.0, 1.0, 3.0], [1.0, 1.0, 1.0, 1.0]], device=DEV)
    ids = _i32([0, 1, 0, 9, 3])
    cu = _i32([0, 4, 5, 5])
    S.repeat_penalty(lg, ids, cu, torch.tensor([2.0, 3.0, 1.5], device=DEV))
    want = torch.stack([P.apply_repeat_penalty(torch.tensor([2.0, -2.0, 1.0, 3.0]), [0, 1, 0, 9], 2.0),
                        P.apply_repeat_penalty(torch.tensor([2.0, -2.0, 1.0, 3.0]), [3], 3.0),
                        torch.ones(4)])
    assert torch.allclose(lg.cpu(), want, atol=1e-6)


def test_cpu_tensors_are_refused(K):
    with pytest.raises(RuntimeError, match="GPU"):
        K.gemm_plain(torch.zeros(2, 2), torch.zeros(2, 2), torch.zeros(2, 2))


# ---------------------------------------------------------------- matrix-core products
@pytest.mark.parametrize("b,v", [(1, 7), (5, 1000), (8, 262208), (3, 4099)])
def test_token_logprob(S, b, v):
    """log softmax at one entry of each row, rows with -inf entries and a row strides apart among them."""
    g = torch.Generator().manual_seed(b + v)
    wide = (torch.randn(b, v + 5, generator=g) * 4).to(DEV)
    logits = wide[:, :v]
    logits[0, : v // 2] = float("-inf")
    toks = torch.randint(v // 2, v, (b,), generator=g).to(torch.int32).to(DEV)
    out = torch.full((b,), float("nan"), device=DEV)
    S.token_logprob(logits, toks, out)
    ref = torch.log_softmax(logits.double(), -1)[torch.arange(b), toks.long()]
    assert torch.allclose(out.double(), ref, atol=2e-5, rtol=0)
    if v > 2:                                               # an entry that is -inf has probability 0
        S.token_logprob(logits, torch.zeros(b, dtype=torch.int32, device=DEV), out)
        assert float(out[0]) == float("-inf")


@pytest.fixture(scope="module")
def G():
    from agave_amd.ops import gemm_mfma
    return gemm_mfma


@pytest.mark.parametrize("m", [1, 3, 16, 17, 40, 64])
@pytest.mark.parametrize("n,k", [(53, 72), (256, 2560), (1000, 96), (4100, 136), (160, 10240)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_gemm_skinny(G, m, n, k, out_dtype):
    g = torch.Generator().manual_seed(m * 1000 + n + k)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
    packed = G.pack_weight(w.to(DEV))
    out = torch.full((m, n), float("nan"), dtype=out_dtype, device=DEV)
    G.skinny(x.to(DEV), packed, out, n)
    ref = x.double() @ w.double().T
    scale = float(ref.abs().max())
    tol = 2e-5 * scale * math.sqrt(k / 64) if out_dtype == torch.float32 else 6e-3 * scale
    assert float((out.cpu().double() - ref).abs().max()) <= tol


@pytest.mark.parametrize("m,ff,k", [(1, 192, 64), (8, 1000, 96), (33, 10240, 256), (64, 20, 40)])
def test_gemm_skinny_geglu(G, m, ff, k):
    g = torch.Generator().manual_seed(ff + m)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(2 * ff, k, generator=g) * 0.2).bfloat16()
    packed = G.pack_weight(w.to(DEV), interleave_ff=ff)
    out = torch.full((m, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    G.skinny(x.to(DEV), packed, out, ff, epilogue=1)
    gu = x.double() @ w.double().T
    ref = P.gelu_tanh(gu[:, :ff]) * gu[:, ff:]
    assert float((out.cpu().double() - ref).abs().max()) <= 8e-3 * float(ref.abs().max())


@pytest.mark.parametrize("m,n,k,slices", [(8, 160, 10240, 3), (1, 53, 4104, 2), (16, 256, 2560, 5), (40, 100, 1096, 2)])
def test_gemm_skinny_in_slices(G, m, n, k, slices):
    """The product shared out along its columns: the 32-bit slices add up to it; runs of columns of
    unequal length, and a last one that ends inside a tile."""
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
    packed = G.pack_weight(w.to(DEV))
    out = torch.full((slices, m, n), float("nan"), device=DEV)
    G.skinny_slices(x.to(DEV), packed, out, n)
    ref = x.double() @ w.double().T
    assert float((out.cpu().double().sum(0) - ref).abs().max()) <= 2e-5 * float(ref.abs().max()) * math.sqrt(k / 64)
    assert float(out[0].abs().max()) > 0 and float(out[-1].abs().max()) > 0
    with pytest.raises(ValueError):
        G.skinny_slices(x.to(DEV), packed, out.bfloat16(), n)
    assert G.slices_for(8, 2560, 10240) > 1 and G.slices_for(8, 10240, 2560) == 1 and G.slices_for(65, 2560, 10240) == 1


@pytest.mark.parametrize("m,n,k,epi", [(1, 4096, 2560, 0), (1, 10240, 2560, 1), (1, 1000, 5376, 1), (1, 53, 200, 0),
                                       (1, 40, 72, 1), (1, 130, 3080, 0), (1, 96, 6144, 0), (1, 8192, 3840, 0),
                                       (1, 21504, 5376, 1), (1, 4100, 4104, 0), (1, 40000, 64, 0), (1, 36, 72, 1),
                                       (1, 21, 40, 0)])
@pytest.mark.parametrize("branch", ["none", "bf16", "f32", "slices", "slices_unnormed", "slices11", "slices2"])
def test_product_of_one_token_that_makes_its_own_normalised_row(G, m, n, k, epi, branch):
    """out = rmsnorm(h + post(branch)) W^T (or its GeGLU) for one row, h + post(branch) going
    to other memory: against the same written out in 64-bit, with the normalised rows rounded to
    bfloat16 as the kernel rounds them.  The gains differ per column and the branch is large against
    h, so that a gain or a norm left out, or applied in the wrong place, shows; memory beside the
    outputs must stay as it was."""
    assert G.normed_ok(m, n, k, epi)
    g = torch.Generator().manual_seed(m * 7 + n + k + len(branch))
    h = torch.randn(m, k, generator=g) * 2
    pre_gain, post_gain = torch.rand(k, generator=g) + 0.5, torch.rand(k, generator=g) * 2 + 0.5
    pre_eps, post_eps = 1e-3, 0.5
    rows = 2 * n if epi else n
    w = (torch.randn(rows, k, generator=g) * 0.1).bfloat16()
    packed = G.pack_weight(w.to(DEV), interleave_ff=n if epi else 0)
    b = b_sum = None
    if branch == "bf16":
        b = (torch.randn(m, k, generator=g) * 5).bfloat16()
        b_sum = b.double()
    elif branch == "f32":
        b = torch.randn(m, k, generator=g) * 5
        b_sum = b.double()
    elif branch.startswith("slices"):
        # (two slices are asked for ahead of the weights, or eight when there are more than two; others follow)
        b = torch.randn({"slices11": 11, "slices2": 2}.get(branch, 5), m, k, generator=g) * 3
        b_sum = b.double().sum(0)
    with_post = branch not in ("none", "slices_unnormed")
    hd = h.double()
    if b_sum is not None:
        if with_post:
            hd = hd + b_sum / torch.sqrt((b_sum * b_sum).mean(-1, keepdim=True) + post_eps) * post_gain.double()
        else:
            hd = hd + b_sum
    x = (hd / torch.sqrt((hd * hd).mean(-1, keepdim=True) + pre_eps) * pre_gain.double()).bfloat16().double()
    y = x @ w.double().T
    ref = P.gelu_tanh(y[:, :n]) * y[:, n:] if epi else y

    h_dev = h.to(DEV)
    h_out = torch.full((m + 1, k), 7.0, device=DEV)
    out = torch.full((m + 1, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    G.row_normed(h_dev, h_out[:m] if b is not None else None, b.to(DEV) if b is not None else None,
                    post_gain.to(DEV) if with_post else None, post_eps, pre_gain.to(DEV), pre_eps, packed, out[:m], n, epi)
    scale = float(ref.abs().max())
    assert float((out[:m].cpu().double() - ref).abs().max()) <= 8e-3 * scale
    assert torch.equal(h_dev.cpu(), h), "the rows that were read are not touched"
    if b is not None:
        assert float((h_out[:m].cpu().double() - hd).abs().max()) <= 2e-5 * float(hd.abs().max())
    else:
        assert float(h_out[:m].min()) == 7.0
    assert float(h_out[m].min()) == 7.0 and float(h_out[m].max()) == 7.0 and bool(torch.isnan(out[m].float()).all())


def test_product_of_one_token_refuses_what_it_cannot_do(G):
    assert not G.normed_ok(2, 4096, 2560, 0) and not G.normed_ok(1, 4096, 6152, 0) and not G.normed_ok(1, 4096, 2564, 0)
    assert not G.normed_ok(1, 262208, 2560, 0)            # (a workgroup would take more row blocks than its LDS holds sums for)
    k, n = 64, 32
    w = G.pack_weight(torch.zeros(n, k, dtype=torch.bfloat16, device=DEV))
    h = torch.zeros(1, k, device=DEV)
    gain = torch.ones(k, device=DEV)
    out = torch.empty(1, n, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError, match="of its own"):
        G.row_normed(h, h, torch.zeros(1, k, device=DEV), None, 0.0, gain, 1e-6, w, out, n)      # the sum in place
    with pytest.raises(ValueError):
        G.row_normed(torch.zeros(3, k, device=DEV), None, None, None, 0.0, gain, 1e-6, w, torch.empty(3, n, dtype=torch.bfloat16, device=DEV), n)
    with pytest.raises(ValueError):
        G.row_normed(h, None, None, None, 0.0, gain, 1e-6, w, out.float(), n)


def test_product_of_many_shapes(G):
    """Shapes drawn at random (fixed seed) across the kernels' cuts: tokens from 1 to 700, rows and
    columns that are multiples of nothing in particular (columns a multiple of 8, which the packed
    product requires), plain and sliced; each against a 64-bit product."""
    rng = np.random.default_rng(7)
    for case in range(48):
        m = int(rng.choice([1, 3, 8, 15, 16, 17, 31, 33, 48, 63, 64, 65, 100, 129, 255, 257, 400, 700]))
        n = int(rng.integers(1, 6000))
        k = 8 * int(rng.integers(1, 700))
        g = torch.Generator().manual_seed(case)
        x = torch.randn(m, k, generator=g).bfloat16()
        w = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
        packed = G.pack_weight(w.to(DEV))
        ref = x.double() @ w.double().T
        scale = float(ref.abs().max()) + 1e-6
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        G.product(x.to(DEV), packed, out, n)
        assert float((out.cpu().double() - ref).abs().max()) <= 6e-3 * scale, (case, m, n, k)
        z = G.slices_for(m, n, k)
        if z > 1:
            parts = torch.full((z, m, n), float("nan"), device=DEV)
            G.skinny_slices(x.to(DEV), packed, parts, n)
            assert float((parts.cpu().double().sum(0) - ref).abs().max()) <= 2e-5 * scale * math.sqrt(k / 64), (case, m, n, k, z)


def test_gemm_skinny_refuses_what_it_cannot_do(G):
    w = G.pack_weight(torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV))
    out = torch.empty(65, 32, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(Exception, match="64"):
        G.skinny(torch.zeros(65, 64, dtype=torch.bfloat16, device=DEV), w, out, 32)
    with pytest.raises(ValueError):
        G.skinny(torch.zeros(4, 60, dtype=torch.bfloat16, device=DEV), w, out[:4], 32)   # K no multiple of 8


@pytest.mark.parametrize("m,nh,hd,splits,n", [(8, 8, 256, 6, 2560), (1, 8, 256, 64, 2560), (16, 32, 128, 4, 5376),
                                              (3, 6, 64, 2, 100), (5, 16, 256, 3, 3840), (2, 4, 96, 9, 250),
                                              (13, 20, 128, 5, 72), (16, 8, 256, 11, 512), (1, 16, 256, 17, 3840)])
def test_product_of_the_decode_attention_s_partial_results(G, m, nh, hd, splits, n):
    """The output projection that merges the splits' partial results itself, against the merge
    written out (with its rows rounded to bfloat16, as the separate merge kernel leaves them) and an
    ordinary product.  Some splits are empty (reference -inf, sum 0), as behind a window's edge."""
    g = torch.Generator().manual_seed(m * 1000 + nh + splits)
    part_o = torch.randn(m, nh, splits, hd, generator=g)
    ref_m = torch.randn(m, nh, splits, generator=g) * 3
    sums = torch.rand(m, nh, splits, generator=g) * 30 + 0.5
    empty = torch.rand(m, nh, splits, generator=g) < 0.2
    empty[:, :, 0] = False                                   # every row keeps a split
    if m > 1:
        empty[1, 0, :] = True                                # but one: no key at all gives zeros
    ref_m[empty], sums[empty] = float("-inf"), 0.0
    part_o[empty] = 0.0
    part_ml = torch.stack([ref_m, sums], dim=-1).contiguous()
    runs = G.partials_runs(m, nh, hd, splits)
    assert 1 <= runs <= 8 and nh % runs == 0
    w = (torch.randn(n, nh * hd, generator=g) * 0.05).bfloat16()
    packed = G.pack_weight(w.to(DEV))
    out = torch.full((runs, m, n), float("nan"), device=DEV)
    G.product_of_partials(part_o.to(DEV), part_ml.to(DEV), packed, out, n)
    mx = ref_m.double().max(dim=-1, keepdim=True).values
    f = torch.where(torch.isinf(ref_m), torch.zeros_like(ref_m, dtype=torch.float64), torch.exp(ref_m.double() - mx))
    f = torch.nan_to_num(f, nan=0.0)
    l = (sums.double() * f).sum(-1)
    x = (part_o.double() * f[..., None]).sum(2) / torch.where(l > 0, l, torch.ones_like(l))[..., None]
    x = torch.where((l > 0)[..., None], x, torch.zeros_like(x)).reshape(m, nh * hd).bfloat16().double()
    ref = x @ w.double().T
    got = out.cpu().double()
    assert torch.isfinite(got).all()
    scale = float(ref.abs().max())
    # a merged value within rounding of a bfloat16 step's middle may round the other way: 2^-8 of one term
    assert float((got.sum(0) - ref).abs().max()) <= 3e-3 * scale
    # each slice is the product over its own run of heads
    cols = nh * hd // runs
    for r in range(runs):
        part = x[:, r * cols:(r + 1) * cols] @ w.double()[:, r * cols:(r + 1) * cols].T
        assert float((got[r] - part).abs().max()) <= 3e-3 * scale, r


def test_product_of_partial_results_refuses_what_it_cannot_do(G):
    assert G.partials_runs(17, 8, 256, 4) == 0          # more than one tile of tokens
    assert G.partials_runs(4, 8, 48, 4) == 0            # heads that are no whole k-steps of 32 columns
    assert G.partials_runs(4, 8, 256, 1) == 0           # nothing to merge
    assert G.partials_runs(16, 32, 128, 65) == 0        # more splits than the kernel merges
    with pytest.raises(ValueError, match="no kernel"):
        G.product_of_partials(torch.zeros(17, 8, 4, 256, device=DEV), torch.zeros(17, 8, 4, 2, device=DEV),
                              G.pack_weight(torch.zeros(32, 2048, dtype=torch.bfloat16, device=DEV)),
                              torch.zeros(8, 17, 32, device=DEV), 32)


# ---------------------------------------------------------------- matrix-core attention over packed pages
class _FakeStep:
    """What the attention op reads of a step."""

    def __init__(self, lens, queries_from, window):
        from agave_amd.parts import Workspace
        self.pos0 = [queries_from(L) for L in lens]
        self.n_new = [L - p for L, p in zip(lens, self.pos0)]
        self.n_seqs = len(lens)
        self.n_tokens = sum(self.n_new)
        self.max_new = max(self.n_new)
        cu = [0]
        for n in self.n_new:
            cu.append(cu[-1] + n)
        self.cu_dev = _i32(cu)
        self.tok_seq = _i32([b for b, n in enumerate(self.n_new) for _ in range(n)])
        self.tok_pos = _i32([p + i for p, n in zip(self.pos0, self.n_new) for i in range(n)])
        self.workspace = Workspace(torch.device(DEV))
        self.fixed_span = None

    @property
    def is_decode(self):
        return self.max_new == 1

    def page_span(self, window):
        span = 1
        for p0, n in zip(self.pos0, self.n_new):
            p = p0 + n - 1
            lo = max(0, p - window + 1) if window is not None else 0
            span = max(span, p // 64 - lo // 64 + 1)
        return span


def _mfma_attn_case(K, nh, nkv, hd, lens, window, scale, decode, seed=0, boost=None, last_row_only=False, fused=False):
    """Keys and values go into packed pages through the q/k kernel (no norm, no rotation); then
    either every position is a query (prefill) or only each sequence's last one (decode)."""
    from agave_amd.ops import attention_mfma
    g = torch.Generator().manual_seed(seed)
    hd_k = (hd + 31) // 32 * 32
    n_pages = sum((L + 63) // 64 for L in lens) + 2
    kp = torch.zeros(n_pages, nkv, 64, hd_k, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros(n_pages, nkv, hd, 64, dtype=torch.bfloat16, device=DEV)
    perm = torch.randperm(n_pages, generator=g).tolist()
    width = max((L + 63) // 64 for L in lens)
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    ks, vs, qs = [], [], []
    for b, L in enumerate(lens):
        k = torch.randn(L, nkv, hd, generator=g).bfloat16()
        v = torch.randn(L, nkv, hd, generator=g).bfloat16()
        q = torch.randn(L, nh, hd, generator=g).bfloat16()
        if boost is not None:
            k = (k.float() - k.float().mean(dim=-1, keepdim=True)).bfloat16()
            k[boost] = 1.0
            q[L - 1] = 20.0 / (hd * scale)
        for i in range((L + 63) // 64):
            table[b, i] = perm.pop()
        ks.append(k); vs.append(v); qs.append(q)
    table, base = table.to(DEV), _i32([0] * len(lens))
    seq_all = _i32([b for b, L in enumerate(lens) for _ in range(L)])
    pos_all = _i32([i for L in lens for i in range(L)])
    k_all = torch.cat(ks).reshape(-1, nkv * hd).to(DEV)
    v_all = torch.cat(vs).reshape(-1, nkv * hd).to(DEV)
    K.qk_norm_rope_kv(None, k_all, v_all, None, None, None, 0.0, 0.0, None, 1.0, seq_all, pos_all, kp, vp, table, base,
                      0, nkv, hd, packed=True)
    step = _FakeStep(lens, (lambda L: L - 1) if decode else (lambda L: 0), window)
    q_sel = torch.cat([q[p0:] for q, p0 in zip(qs, step.pos0)]).reshape(-1, nh * hd).to(DEV)
    out = torch.full_like(q_sel, float("nan"))
    if fused:       # the decode kernel that also takes the new token's q and k: here it appends nothing
        attention_mfma.decode_fused(q_sel, None, None, out, None, None, 0.0, 0.0, None, 1.0, kp, vp, table, base, step,
                                    nh, nkv, hd, scale, window)
    else:
        attention_mfma.attention(q_sel, out, kp, vp, table, base, step, nh, nkv, hd, scale, window)
    if last_row_only and not decode:
        refs = []                                           # the caller checks rows of its choice
    elif last_row_only:
        refs = [_last_row_attention(q.double(), k.double(), v.double(), scale, window) for q, k, v in zip(qs, ks, vs)]
    else:
        refs = [P.attention_core(q.double(), k.double(), v.double(), scale, window)[p0:]
                for q, k, v, p0 in zip(qs, ks, vs, step.pos0)]
    return out.cpu().double().view(-1, nh, hd), (torch.cat(refs) if refs else (qs, ks)), vs


def _last_row_attention(q, k, v, scale, window):
    """The last position's attention alone, as a library softmax over its keys: what the whole
    table of scores would cost too much for at tens of thousands of keys.  q [L, nh, hd], k, v [L, nkv, hd]."""
    L, nh, _ = q.shape
    group = nh // k.shape[1]
    first = max(0, L - window) if window is not None else 0
    out = torch.empty(1, nh, v.shape[-1], dtype=torch.float64)
    for h in range(nh):
        scores = (k[first:, h // group] @ q[L - 1, h]) * scale
        out[0, h] = torch.softmax(scores, 0) @ v[first:, h // group]
    return out


@pytest.mark.parametrize("decode", [True, False])
@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 64, None), (6, 1, 16, 70), (3, 3, 48, 300), (8, 4, 256, 64),
                                              (2, 1, 128, None), (20, 1, 32, 129), (8, 2, 96, 1)])
def test_attn_mfma(K, decode, nh, nkv, hd, window):
    got, ref, _ = _mfma_attn_case(K, nh, nkv, hd, [1, 77, 300, 64, 65], window, 0.21 * (16 / hd) ** 0.5, decode)
    assert torch.isfinite(got).all()
    assert torch.allclose(got, ref, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("decode", [True, False])
def test_attn_mfma_long_sequences_split_over_workgroups(K, decode):
    from agave_amd.ops import attention_mfma
    assert attention_mfma.split_plan(40, 4)[0] > 1          # the decode launch below is split
    got, ref, _ = _mfma_attn_case(K, 4, 2, 128, [2500, 1031], None, 0.05, decode, seed=3)
    assert torch.allclose(got, ref, atol=2e-2, rtol=2e-2)
    got, ref, _ = _mfma_attn_case(K, 4, 2, 128, [2500, 1031], 1024, 0.05, decode, seed=4)
    assert torch.allclose(got, ref, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("nh,nkv,hd,lens,window", [(8, 4, 256, [20000, 9001, 100], None), (8, 4, 256, [20000, 9001], 1024),
                                                   (5, 1, 80, [33000], None), (2, 2, 64, [70000, 3], 4097)])
def test_attn_mfma_decode_over_tens_of_thousands_of_keys(K, nh, nkv, hd, lens, window):
    """Hundreds of pages a sequence, beside a short one: every share of the pages and their merge,
    with key 3 made to win in one pass (the furthest key there is) and random scores in the other."""
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn(9, n, 8, generator=g).double() for n in (4, 2, 2))
    for w in (None, 5):                                     # the helper is the plain function's last row
        assert torch.allclose(_last_row_attention(q, k, v, 0.3, w), P.attention_core(q, k, v, 0.3, w)[-1:], atol=1e-12)
    got, ref, _ = _mfma_attn_case(K, nh, nkv, hd, lens, window, 0.3 * (16 / hd) ** 0.5, True, seed=11, last_row_only=True)
    assert torch.isfinite(got).all()
    assert torch.allclose(got, ref, atol=2e-2, rtol=2e-2)
    if window is None:
        got, ref, vs = _mfma_attn_case(K, nh, nkv, hd, lens, None, 0.5, True, seed=12, boost=3, last_row_only=True)
        assert torch.allclose(got, ref, atol=2e-2, rtol=2e-2)
        assert torch.allclose(got[0, 0], vs[0][3, 0].double(), atol=2e-2)


@pytest.mark.parametrize("nh,nkv,hd,L,window", [(4, 2, 128, 20000, None), (8, 4, 256, 9001, 1024), (3, 1, 48, 40000, 5000)])
def test_attn_mfma_prefill_of_tens_of_thousands_of_tokens(K, nh, nkv, hd, L, window):
    """A prompt of hundreds of pages in one step; rows at the start, at page edges, in the middle
    and at the end are compared, each as the last row of the sequence that ends with it."""
    scale = 0.3 * (16 / hd) ** 0.5
    got, (qs, ks), vs = _mfma_attn_case(K, nh, nkv, hd, [L], window, scale, False, seed=13, last_row_only=True)
    assert torch.isfinite(got).all()
    for r in (0, 63, 64, 1023, 1024, L // 2 + 7, L - 65, L - 1):
        ref = _last_row_attention(qs[0][:r + 1].double(), ks[0][:r + 1].double(), vs[0][:r + 1].double(), scale, window)
        assert torch.allclose(got[r:r + 1], ref, atol=2e-2, rtol=2e-2), r


@pytest.mark.parametrize("nh,nkv,hd,lens,window", [(4, 2, 128, [1500], None), (4, 2, 128, [1500], 1024),
                                                   (8, 4, 256, [700, 300], None), (2, 2, 64, [1100, 64, 1], 600)])
def test_attn_mfma_prefill_blocks_shared_among_workgroups(K, nh, nkv, hd, lens, window):
    """A prompt with few blocks of positions: the blocks with a long reach are cut into pieces
    that go to workgroups of their own, and a second pass merges what they leave."""
    from agave_amd.ops import attention_mfma
    hw = 2 if nh // nkv >= 2 else 1
    plan = attention_mfma.plan_prefill_items([0] * len(lens), lens, window, (8 // hw) * 16, nkv, nh, hd)
    assert plan[2] > 1 and (plan[1] > 1).any() and (plan[1] == 1).any()      # some blocks in pieces, some whole
    got, ref, _ = _mfma_attn_case(K, nh, nkv, hd, lens, window, 0.3 * (16 / hd) ** 0.5, False, seed=7)
    assert torch.isfinite(got).all()
    assert torch.allclose(got, ref, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("how,hd", [(how, hd) for how in ("decode", "fused decode", "prefill") for hd in (32, 64, 128, 256)
                                    if not (how == "fused decode" and hd == 32)])      # (the fused kernel: 64, 128, 256)
def test_attn_mfma_far_key_and_window_edge(K, how, hd):
    """Key 3 of 700 is made to win every score of the last query; a window that ends just before
    it must lose it and one that just includes it must keep it.  Head size 32 takes the general
    kernels, 64 to 256 the fast ones (and the decode kernel that also handles the new token)."""
    kw = dict(decode=how != "prefill", fused=how == "fused decode", seed=1, boost=3)
    scale = 0.5 * (32 / hd) ** 0.5
    got, ref, vs = _mfma_attn_case(K, 2, 1, hd, [700], None, scale, **kw)
    assert torch.allclose(got[-1, 0], vs[0][3, 0].double(), atol=2e-2)
    got_w, _, _ = _mfma_attn_case(K, 2, 1, hd, [700], 696, scale, **kw)      # key 3 just outside
    assert not torch.allclose(got_w[-1, 0], vs[0][3, 0].double(), atol=1e-1)
    got_e, _, _ = _mfma_attn_case(K, 2, 1, hd, [700], 697, scale, **kw)      # just inside
    assert torch.allclose(got_e[-1, 0], vs[0][3, 0].double(), atol=2e-2)
    # the same at a window's edge that falls on a page's edge and one row either side of it
    for window, inside in ((700 - 64, False), (700 - 63, False), (700 - 3, True), (700 - 4, False)):
        got_p, _, _ = _mfma_attn_case(K, 2, 1, hd, [700], window, scale, **kw)
        assert torch.allclose(got_p[-1, 0], vs[0][3, 0].double(), atol=2e-2) == inside, window


# the last three shapes take the 128 x 128, 128 x 256 and 256 x 256 tiles, the others the 64 x 128 one; the
# shapes with few tiles and many columns are shared out along the columns (2, 5, 3 and 7 partial sums)
@pytest.mark.parametrize("m,n,k", [(65, 53, 72), (300, 256, 2560), (100, 250, 2560), (70, 200, 1560), (65, 2560, 10240),
                                   (257, 1000, 96), (2048, 300, 136), (130, 4100, 64),
                                   (1000, 4096, 96), (2048, 4090, 64), (1024, 10240, 72),
                                   # many stages (the loads run several stages ahead of the multiplications): each tile
                                   (300, 2000, 1000), (600, 5000, 1000), (1024, 5120, 1000), (1024, 10240, 1000),
                                   # 640 tiles: two rounds of 256 x 256 tiles and the last rows in tiles of half the height
                                   (2048, 20470, 64),
                                   # 320 tiles: one round and the last rows in tiles of a quarter of the size
                                   (1024, 20470, 64)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_gemm_tiled(G, m, n, k, out_dtype):
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
    packed = G.pack_weight(w.to(DEV))
    out = torch.full((m, n), float("nan"), dtype=out_dtype, device=DEV)
    G.product(x.to(DEV), packed, out, n)
    ref = x.double() @ w.double().T
    scale = float(ref.abs().max())
    tol = 2e-5 * scale * math.sqrt(k / 64) if out_dtype == torch.float32 else 6e-3 * scale
    assert float((out.cpu().double() - ref).abs().max()) <= tol


@pytest.mark.parametrize("m,n,k,slices", [
    (2048, 2560, 10240, 3),     # 160 tiles of 128 x 256: three slices, which run as 240 tiles of 256 x 256
    (4096, 2560, 10240, 1),     # 160 tiles of 256 x 256: one product
    (2000, 2552, 10248, 3),     # ragged edges
    (8192, 640, 10240, 3),      # 160 tiles of 128 x 256 whose slices in 256 x 256 would be 288: they stay 480 of 128 x 256
    (2048, 2560, 2048, 1),      # few columns: one product
    (1024, 2560, 10240, 3),     # a shorter prompt: 80 tiles of 128 x 256 in three slices
    (768, 2560, 10240, 4),      # 60 tiles in four
    (1024, 2560, 2048, 1),      # 80 tiles, but too few columns for a slice
    (300, 200, 4096, 8),        # next to no tiles of 64 x 128 (12): as many slices of those as leave eight stages each
    (256, 2560, 10240, 3),      # a short prompt: 80 tiles of 64 x 128 in three slices, one round of workgroups
    (384, 2560, 10240, 2),      # 120 tiles in two
    (130, 2560, 2048, 3),       # few columns: the slices keep six stages each (32 stages: five slices; 80 tiles: three)
    (100, 2560, 2048, 5),       # 40 tiles of 32 stages: five slices
    (256, 3840, 4096, 2),       # 120 tiles of 64 x 128 in two slices
    (384, 3840, 4096, 1),       # more tokens: 4,096 columns in slices of 128 x 256 tiles lose to the one product
    (200, 640, 320, 1)])        # five stages in all: one product
def test_gemm_tiled_in_slices(G, m, n, k, slices):
    """A product of many tokens whose tiles fill the compute units badly comes as 32-bit slices
    that add up to it, for a reader that adds them."""
    z = G.tiled_slices_for(m, n, k)
    assert z == slices
    if z == 1:
        return
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
    packed = G.pack_weight(w.to(DEV))
    out = torch.full((z, m, n), float("nan"), dtype=torch.float32, device=DEV)
    G.tiled_slices(x.to(DEV), packed, out, n)
    ref = x.to(DEV).double() @ w.to(DEV).double().T
    got = out.double().sum(0)
    assert float((got - ref).abs().max()) <= 2e-5 * float(ref.abs().max()) * math.sqrt(k / 64)
    assert float(out[0].abs().max()) > 0 and float(out[z - 1].abs().max()) > 0


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("m,n,k,z", [(300, 520, 1024, 1), (70, 200, 4096, 5), (513, 1000, 1544, 3), (256, 2560, 2048, 8)])
def test_gemm_tiled_every_tile_shape_in_slices(G, tile, m, n, k, z):
    """Each tile shape alone (256 x 256, 128 x 256, 128 x 128, 64 x 128), as one product and in
    slices, whatever the library's own choice for these sizes would be."""
    g = torch.Generator().manual_seed(m + n + k + tile)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
    packed = G.pack_weight(w.to(DEV))
    ref = x.double() @ w.double().T
    out = torch.full((z, m, n), float("nan"), dtype=torch.float32, device=DEV)
    G.tiled_slices_as(x.to(DEV), packed, out, n, tile)
    assert float((out.double().sum(0).cpu() - ref).abs().max()) <= 2e-5 * float(ref.abs().max()) * math.sqrt(k / 64)
    whole = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    G.tiled_as(x.to(DEV), packed, whole, n, tile)
    assert float((whole.double().cpu() - ref).abs().max()) <= 6e-3 * float(ref.abs().max())


# 32-bit products in pieces on the bfloat16 instructions: every tile shape, its last rows and columns broken, stages of 32 columns
# broken, one of them, as many as slices and more; rows that lie apart; values next to the largest float, which round to an infinity.
@pytest.mark.parametrize("tile", [(128, 128), (64, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("m,n", [(17, 5), (64, 64), (129, 65), (200, 258)])
@pytest.mark.parametrize("k,z", [(4, 1), (36, 2), (64, 1), (260, 8), (1028, 4)])
def test_gemm_slices(K, tile, m, n, k, z):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k + 8, device=DEV, generator=g)[:, 4:4 + k]
    w = torch.randn(n, k + 4, device=DEV, generator=g)[:, :k]
    for scale in (1.0, 2.0 ** -40, 2.0 ** 60):              # (pieces of 2^-40 and less are still whole numbers of the smallest float)
        parts = torch.full((z, m, n), float("nan"), device=DEV)
        K.gemm_slices(x * scale if scale != 1.0 else x, w, parts, tile)
        ref, size = x.double() * scale @ w.double().T, (x.double() * scale).abs() @ w.double().abs().T
        # a piece's rest is below 2^-23 of a product (three products of the nine are left out), an addition below 2^-24 of the sum
        assert bool(((parts.double().sum(0) - ref).abs() <= (k + 2) * 2.0 ** -24 * size).all())
    x[1, k - 1], x[m - 1, 0], w[2, 1], w[n - 1, k - 2] = float("nan"), float("inf"), float("-inf"), 3.4e38
    x[3] *= 1e-3
    parts = torch.full((z, m, n), float("nan"), device=DEV)
    K.gemm_slices(x, w, parts, tile)
    got, want = parts.double().sum(0), x.double() @ w.double().T
    plain = torch.ones(m, n, dtype=torch.bool, device=DEV)
    plain[[1, m - 1]], plain[:, [2, n - 1]] = False, False
    assert bool(got[plain].isfinite().all()) and bool(got[1].isnan().all())
    assert not bool(got[m - 1].isfinite().any()) and not bool(got[:, 2].isfinite().any())
    assert abs(float(got[3, n - 1] / want[3, n - 1]) - 1) <= (k + 2) * 2.0 ** -24       # (the large product outweighs the others)


# Small floats have bits below the last one that a bfloat16 piece can hold (2^-133): from some 2^-110 on either operand's, down to the
# numbers without an exponent, and beside them in the same row some whose pieces leave 32 bits when they are made larger.
@pytest.mark.parametrize("tile", [(128, 128), (64, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("power", [-100, -112, -118, -126, -140])
@pytest.mark.parametrize("small", ["x", "w", "a row of either"])
def test_gemm_slices_of_small_floats(K, tile, power, small):
    m, n, k, z = 70, 136, 260, 2
    g = torch.Generator(device=DEV).manual_seed(-power)
    x, w = torch.randn(m, k, device=DEV, generator=g), torch.randn(n, k, device=DEV, generator=g)
    down = lambda t: (t.double() * 2.0 ** power).float()
    if small == "x":
        x = down(x)
    elif small == "w":
        w = down(w)
    else:
        x[5], w[7, ::2] = down(x[5]), down(w[7, ::2])
        x[9, 3], w[11, 4] = 2.0 ** 110, -2.0 ** 119
    parts, plain = torch.full((z, m, n), float("nan"), device=DEV), torch.empty(m, n, device=DEV)
    K.gemm_slices(x, w, parts, tile)
    K.gemm_plain(x, w, plain)
    ref, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # as above, and a product or a sum below 2^-126 is rounded to a whole number of 2^-149
    off = (k + 2) * 2.0 ** -24 * size + (k + z) * 2.0 ** -150
    assert bool(((parts.double().sum(0) - ref).abs() <= off).all()) and bool(((plain.double() - ref).abs() <= off).all())
    assert float((parts.double().sum(0) - ref)[5].norm()) <= 1.1 * float((plain.double() - ref)[5].norm())


@pytest.mark.parametrize("m,n,k", [(33, 2048, 2048), (64, 10752, 2048), (100, 512, 2048), (200, 2048, 5376), (700, 3072, 2048), (17, 2304, 9216)])
def test_gemm_in_slices_is_as_exact_as_whole(K, m, n, k):
    """Where a product is made in slices its error against 64 bits is no larger than that of the kernels of the 32-bit instructions
    (1.0 to 2.1e-7 of the result over these sizes, 2.9 to 5.7e-7 there)."""
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x, w = torch.randn(m, k, device=DEV, generator=g), torch.randn(n, k, device=DEV, generator=g)
    z = K.gemm_slices_for(x, w)
    assert z > 1 and K.gemm_slices_for(x[:, 1:], w[:, 1:]) == 1 and K.gemm_slices_for(x.bfloat16(), w) == 1
    parts, out, plain = torch.empty(z, m, n, device=DEV), torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    K.gemm_slices(x, w, parts)
    K.add_slices(parts, out)
    K.gemm_plain(x, w, plain)
    ref = x.double() @ w.double().T
    of = lambda c: float((c.double() - ref).pow(2).mean().sqrt() / ref.pow(2).mean().sqrt())
    print(m, n, k, "slices", z, "error", of(out), "whole", of(plain))
    assert of(out) <= 1.1 * of(plain)


# Between the rings of 32 and of 128 rows: three tiles of either kernel a compute unit, their last rows and columns broken.  Two running
# sums an element as in the rings (some 5.7e-7 of the result at 2,048 columns, 8.1e-7 with one; the bound lies between).
@pytest.mark.parametrize("m,n", [(1500, 2050), (510, 5372), (130, 16000), (1536, 2048)])
@pytest.mark.parametrize("k", [4, 36, 2052])
def test_gemm_plain_three_tiles_a_unit(K, m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x, w = torch.randn(m, k + 4, device=DEV, generator=g)[:, :k], torch.randn(n, k, device=DEV, generator=g)
    c = torch.full((m + 1, n + 2), 7.0, device=DEV)
    K.gemm_plain(x, w, c[:m, :n])
    ref = x.double() @ w.double().T
    err = (c[:m, :n].double() - ref).abs()
    assert bool((err <= k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all())
    assert float(err.pow(2).mean().sqrt()) <= 6.8e-7 * float(ref.pow(2).mean().sqrt())
    assert bool((c[m] == 7.0).all()) and bool((c[:, n:] == 7.0).all())


# Columns: one stage of 64 and less, a k-step of 32 missing from the last stage, as many stages as the ring has buffers and
# one more or less, many.  Rows and tokens: a tile of each shape, one more, one less.
@pytest.mark.parametrize("k", [8, 64, 72, 96, 192, 200, 256, 320, 1000])
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("gated", [False, True])
def test_gemm_tile_edges(G, tile, gated, k):
    rows, tokens = G.TILE_SHAPES[tile]
    g = torch.Generator().manual_seed(tile + k)
    for m, n in ((tokens, rows), (tokens + 1, rows + 1), (2 * tokens - 1, 2 * rows - 3), (3, 5)):
        n = (n + 1) // 2 if gated else n
        x = torch.randn(m, k + 24, generator=g).bfloat16().to(DEV)[:, :k]            # (rows further apart than they are long)
        w = (torch.randn(2 * n if gated else n, k, generator=g) * 0.2).bfloat16().to(DEV)
        packed = G.pack_weight(w, interleave_ff=n if gated else 0)
        ref = x.double() @ w.double().T
        if gated:
            ref = P.gelu_tanh(ref[:, :n]) * ref[:, n:]
        out = torch.full((m, n + 3), float("nan"), dtype=torch.bfloat16, device=DEV)
        G.tiled_as(x, packed, out[:, :n], n, tile, epilogue=int(gated))
        # bfloat16 results (half an ulp: 2^-9 of each), of sums in 32 bits whose rounding is far below; gated: of two factors
        assert float((out[:, :n].double() - ref).abs().max()) <= (8e-3 if gated else 6e-3) * float(ref.abs().max())
        assert bool(out[:, n:].isnan().all())
        if gated or tile in G.BF16_ONLY_TILES or m <= 64:            # (slices: more than 64 tokens)
            continue
        whole = torch.full((1, m, n), float("nan"), device=DEV)
        G.tiled_slices_as(x, packed, whole, n, tile)
        assert float((whole[0].double() - ref).abs().max()) <= 2e-5 * float(ref.abs().max()) * math.sqrt(max(k, 64) / 64)


# Whole rounds of 256 x 256 tiles in one launch and the rows behind them in a second one, in tiles of each shape: a last row block that is
# not whole, tokens that are not, and the biases of a gated product, which the second launch reads further on.
@pytest.mark.parametrize("m,n,k", [(500, 41682, 3072), (257, 41692, 3072), (769, 32804, 1024), (769, 24630, 1024), (257, 44254, 3072),
                                   (257, 43668, 3072)])
@pytest.mark.parametrize("gated", [False, True])
def test_gemm_tiled_last_round_in_a_launch_of_its_own(G, m, n, k, gated):
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(m, k, device=DEV, generator=g).bfloat16()
    w = (torch.randn(n, k, device=DEV, generator=g) * 0.05).bfloat16()
    no = n // 2 if gated else n
    form = G.GELU_TANH
    if gated:
        bg, bu = (torch.randn(no, device=DEV, generator=g) for _ in range(2))
        form = form._replace(gate_bias=bg, up_bias=bu)
    out = torch.full((m, no + 3), float("nan"), dtype=torch.bfloat16, device=DEV)
    G.product(x, G.pack_weight(w, interleave_ff=no if gated else 0), out[:, :no], no, epilogue=int(gated), form=form)
    ref = x.float() @ w.float().T
    if gated:
        gate = ref[:, :no] + bg
        ref = P.gelu_tanh(gate) * (ref[:, no:] + bu)
    # (bfloat16 results: half an ulp, 2^-9 of each; gated, of a product of two factors)
    err = (out[:, :no].float() - ref).abs()
    assert float(err.max()) <= (8e-3 if gated else 6e-3) * float(ref.abs().max())
    assert bool((err.max(0).values <= 2.0 ** -7 * ref.abs().max(0).values + 2e-3).all())          # (every column by itself)
    assert bool(out[:, no:].isnan().all())


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("k", [40, 104, 136, 328])
def test_gemm_tile_infinities_stay_theirs(G, tile, k):
    """Whatever stands in a row stays that row's, and what is read in the place of missing columns counts nothing: a row with an
    infinity anywhere gives infinities of the right sign, not NaN."""
    g = torch.Generator().manual_seed(k)
    m, n = 140, 170
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.rand(n, k, generator=g) + 0.5).bfloat16()
    for r, c in enumerate(range(0, k, 8)):
        x[r, c] = math.inf if r % 2 else -math.inf
    marked = (k + 7) // 8
    out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    G.tiled_as(x.to(DEV), G.pack_weight(w.to(DEV)), out, n, tile)
    got = out.cpu().double()
    assert torch.equal(got[:marked], torch.tensor([[math.inf if r % 2 else -math.inf] * n for r in range(marked)], dtype=torch.float64))
    ref = x.double()[marked:] @ w.double().T
    assert float((got[marked:] - ref).abs().max()) <= 6e-3 * float(ref.abs().max())


# Tiles of 64 tokens by 128, 96 and 64 weight rows (160 to 256 workgroups of each make a round that is filled well enough):
# rows that end inside a tile, columns that end inside a stage, fewer stages than the ring has buffers, 17 and 64 tokens, and
# the products of one whole round that fewer tokens take them for.
@pytest.mark.parametrize("m,n,k", [(17, 32760, 72), (64, 32760, 200), (2, 32760, 328), (1, 32768, 64), (16, 32765, 1000),
                                   (33, 20530, 104), (64, 24570, 64), (20, 10750, 456), (63, 10300, 8), (64, 16380, 1096)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32, "gated"])
def test_gemm_tiles_of_64_tokens(G, m, n, k, out_dtype):
    g = torch.Generator().manual_seed(m + n + k)
    gated = out_dtype == "gated"
    n = n // 2 if gated else n
    x = torch.randn(m, k + 8, generator=g).bfloat16().to(DEV)[:, :k]
    w = (torch.randn(2 * n if gated else n, k, generator=g) * 0.1).bfloat16().to(DEV)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16 if gated else out_dtype, device=DEV)
    G.product(x, G.pack_weight(w, interleave_ff=n if gated else 0), out, n, epilogue=int(gated))
    ref = x.double() @ w.double().T
    if gated:
        ref = P.gelu_tanh(ref[:, :n]) * ref[:, n:]
    scale = float(ref.abs().max())
    tol = 2e-5 * scale * math.sqrt(max(k, 64) / 64) if out_dtype == torch.float32 else 8e-3 * scale
    assert float((out.double() - ref).abs().max()) <= tol


# 32-bit results: products of up to 16 tokens share their columns among waves, the tiles and whole products of more tokens do
# not.  Their running sums must not be further off for that; a wave's share is 16 k-steps at the most where the columns are 2,048
# (root mean square some 1.3e-7 of the result, 2.7e-7 as one running sum; the bound lies at the geometric mean).
@pytest.mark.parametrize("m,n", [(17, 32768), (64, 20480), (8, 32768), (64, 16384), (65, 8512), (100, 8192), (300, 2560)])
def test_32_bit_products_round_as_shared_columns_do(G, m, n):
    k = 2048
    g = torch.Generator(device=DEV).manual_seed(m)
    x, w = (torch.randn(r, k, device=DEV, generator=g).bfloat16() for r in (m, n))
    out = torch.empty(m, n, device=DEV)
    G.product(x, G.pack_weight(w), out, n)
    ref = x.double() @ w.double().T
    assert float((out.double() - ref).pow(2).mean().sqrt()) <= 1.9e-7 * float(ref.pow(2).mean().sqrt())


@pytest.mark.parametrize("m,n,k", [(17, 2560, 10240), (64, 2552, 10248), (40, 2560, 2048), (33, 2040, 5384), (64, 4304, 5168)])
def test_gemm_tiles_of_64_tokens_in_slices(G, m, n, k):
    z = G.slices_for(m, n, k)
    assert 1 < z <= 8
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16().to(DEV)
    w = (torch.randn(n, k, generator=g) * 0.1).bfloat16().to(DEV)
    out = torch.full((z, m, n), float("nan"), device=DEV)
    G.skinny_slices(x, G.pack_weight(w), out, n)
    ref = x.double() @ w.double().T
    assert float((out.double().sum(0) - ref).abs().max()) <= 2e-5 * float(ref.abs().max()) * math.sqrt(k / 64)


@pytest.mark.parametrize("m,ff,k", [(70, 192, 64), (513, 1000, 96), (256, 20, 40), (1024, 5120, 1000), (2048, 10236, 64),
                                    (1024, 10236, 64)])
def test_gemm_tiled_geglu(G, m, ff, k):
    g = torch.Generator().manual_seed(ff + m)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(2 * ff, k, generator=g) * 0.2).bfloat16()
    packed = G.pack_weight(w.to(DEV), interleave_ff=ff)
    out = torch.full((m, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    G.product(x.to(DEV), packed, out, ff, epilogue=1)
    gu = x.double() @ w.double().T
    ref = P.gelu_tanh(gu[:, :ff]) * gu[:, ff:]
    assert float((out.cpu().double() - ref).abs().max()) <= 8e-3 * float(ref.abs().max())


def test_embedding_from_a_packed_table(G):
    table = (torch.randn(300, 72) * 0.05).bfloat16()
    packed = G.pack_weight(table.to(DEV))
    toks = [0, 299, 17, 17, 123, 16, 15]
    out = torch.empty(len(toks), 72, dtype=torch.float32, device=DEV)
    G.embed_scale_packed(_i32(toks), packed, math.sqrt(72.0), out, 300)
    assert torch.allclose(out.cpu().double(), P.embed(toks, table.double(), 72), atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("nh,nkv,hd,window,rot", [(8, 4, 256, 64, 128), (4, 2, 64, None, 16), (40, 2, 128, 1000, 64),
                                                  (2, 2, 128, None, 0)])
def test_attn_decode_fused_equals_the_two_kernels(K, nh, nkv, hd, window, rot):
    """The decode kernel that normalises, rotates and caches the new token itself must leave the
    same bits, in the output and in the cache pages, as the q/k kernel followed by the attention
    kernel; appending nothing (k None) must leave the pages alone."""
    from agave_amd.ops import attention as A
    g = torch.Generator().manual_seed(11)
    lens = [1, 64, 65, 300, 1500, 128]                  # positions at a page's first and last row among them
    B = len(lens)
    n_pages = sum((L + 63) // 64 for L in lens) + 1
    width = max((L + 63) // 64 for L in lens)
    perm = torch.randperm(n_pages, generator=g).tolist()
    table = torch.full((B, width), -1, dtype=torch.int32)
    for b, L in enumerate(lens):
        for i in range((L + 63) // 64):
            table[b, i] = perm.pop()
    table, base = table.to(DEV), _i32([0] * B)
    kp0 = torch.randn(n_pages, nkv, 64, hd, generator=g).bfloat16().to(DEV)      # older keys: any values
    vp0 = torch.randn(n_pages, nkv, hd, 64, generator=g).bfloat16().to(DEV)
    q = torch.randn(B, nh * hd, generator=g).bfloat16().to(DEV)
    k = torch.randn(B, nkv * hd, generator=g).bfloat16().to(DEV)
    v = torch.randn(B, nkv * hd, generator=g).bfloat16().to(DEV)
    qg = (1 + 0.2 * torch.randn(hd, generator=g)).to(DEV)
    kg = (1 + 0.2 * torch.randn(hd, generator=g)).to(DEV)
    inv_freq = torch.exp(-torch.arange(rot).float() / max(rot, 1) * 5).to(DEV) if rot else None
    step = _FakeStep(lens, lambda L: L - 1, window)
    scale = 0.3 * (16 / hd) ** 0.5
    outs = []
    for fused in (True, False):
        kp, vp = kp0.clone(), vp0.clone()
        out = torch.full_like(q, float("nan"))
        q_rot = torch.empty_like(q)
        if fused:
            A.qk_attention(q, k, v, q_rot, out, qg, kg, 1e-5, 2e-6, inv_freq, 0.5, kp, vp, table, base, step,
                           nh, nkv, hd, scale, window, True)
        else:
            K.qk_norm_rope_kv(q, k, v, q_rot, qg, kg, 1e-5, 2e-6, inv_freq, 0.5, step.tok_seq, step.tok_pos, kp, vp,
                              table, base, nh, nkv, hd, packed=True)
            A.attention(q_rot, out, kp, vp, table, base, step, nh, nkv, hd, scale, window, True)
        torch.cuda.synchronize()
        outs.append((out, kp, vp))
    assert torch.isfinite(outs[0][0].float()).all()
    for a, b, what in zip(outs[0], outs[1], ("output", "K pages", "V pages")):
        assert torch.equal(a, b), what
    # a run that appends nothing: queries only, pages untouched
    kp, vp = outs[1][1].clone(), outs[1][2].clone()
    out = torch.full_like(q, float("nan"))
    A.qk_attention(q, None, None, torch.empty_like(q), out, qg, kg, 1e-5, 2e-6, inv_freq, 0.5, kp, vp, table, base,
                   step, nh, nkv, hd, scale, window, True)
    assert torch.equal(out, outs[1][0]) and torch.equal(kp, outs[1][1]) and torch.equal(vp, outs[1][2])


# Where the decode kernel can go wrong at the token's own row: every place of it within a unit of 32 keys' registers, windows that
# begin inside a unit, more than four jobs a workgroup, two chunks of heads, tables wider than a wave, with and without columns that
# begin at the reach.  Until the kernel writes it, the row in the page is not a number, so whoever read it from there would be seen.
@pytest.mark.parametrize("from_reach", [True, False])
@pytest.mark.parametrize("nh,nkv,hd,window,lens", [
    (8, 4, 256, None, [1, 2, 4, 5, 13, 16, 17, 18, 29, 32, 33, 49, 64, 65, 96, 128, 161, 700]),
    (8, 4, 256, 40, [1, 16, 17, 33, 40, 41, 57, 64, 100, 129]), (5, 1, 128, None, [3, 20, 31, 95, 320]),
    (18, 1, 64, 100, [1, 21, 32, 101, 230]), (2, 2, 256, None, [4200, 4097, 70]), (2, 1, 128, None, [4200, 33]),
    (4, 2, 64, None, [30, 6000])])
def test_attn_decode_fused_own_row(K, nh, nkv, hd, window, lens, from_reach):
    from agave_amd.ops import attention_mfma as A
    g = torch.Generator().manual_seed(hd + len(lens))
    B, n_pages = len(lens), sum((L + 63) // 64 for L in lens) + 1
    kp = torch.zeros(n_pages, nkv, 64, hd, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros(n_pages, nkv, hd, 64, dtype=torch.bfloat16, device=DEV)
    perm = torch.randperm(n_pages, generator=g).tolist()
    full = torch.full((B, max((L + 63) // 64 for L in lens)), -1, dtype=torch.int32)
    ks, vs, scale = [], [], 0.3 * (16 / hd) ** 0.5
    for b, L in enumerate(lens):
        ks.append(torch.randn(L, nkv, hd, generator=g).bfloat16())
        vs.append(torch.randn(L, nkv, hd, generator=g).bfloat16())
        for i in range((L + 63) // 64):
            full[b, i] = perm.pop()
    k_bad, v_bad = [k.clone() for k in ks], [v.clone() for v in vs]
    for k, v in zip(k_bad, v_bad):
        k[-1], v[-1] = float("nan"), float("nan")
    flat = lambda xs: torch.cat(xs).reshape(-1, nkv * hd).to(DEV)
    K.qk_norm_rope_kv(None, flat(k_bad), flat(v_bad), None, None, None, 0.0, 0.0, None, 1.0,
                      _i32([b for b, L in enumerate(lens) for _ in range(L)]), _i32([i for L in lens for i in range(L)]), kp, vp,
                      full.to(DEV), _i32([0] * B), 0, nkv, hd, packed=True)
    step = _FakeStep(lens, lambda L: L - 1, window)
    table, base = full, [0] * B
    if from_reach:
        step.tables_start_at_reach = True
        base = [max(0, L - window) // 64 if window else 0 for L in lens]
        table = torch.full_like(full, -1)
        for b in range(B):
            table[b, :full.shape[1] - base[b]] = full[b, base[b]:]
    q = torch.randn(B, nh, hd, generator=g).bfloat16()
    out = torch.full((B, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    A.decode_fused(q.reshape(B, -1).to(DEV), flat([k[-1:] for k in ks]), flat([v[-1:] for v in vs]), out, None, None, 0.0, 0.0, None, 1.0,
                   kp, vp, table.to(DEV), _i32(base), step, nh, nkv, hd, scale, window)
    ref = torch.cat([_last_row_attention(q[b][None].expand(L, nh, hd).double(), ks[b].double(), vs[b].double(), scale, window)
                     for b, L in enumerate(lens)])
    # (probabilities and results are rounded to bfloat16, half a unit of 2^-8 each; values are below 5)
    assert torch.allclose(out.cpu().double().view(B, nh, hd), ref, atol=2e-2, rtol=1e-2)
    want_k, want_v = torch.zeros_like(kp), torch.zeros_like(vp)
    K.qk_norm_rope_kv(None, flat(ks), flat(vs), None, None, None, 0.0, 0.0, None, 1.0,
                      _i32([b for b, L in enumerate(lens) for _ in range(L)]), _i32([i for L in lens for i in range(L)]), want_k, want_v,
                      full.to(DEV), _i32([0] * B), 0, nkv, hd, packed=True)
    assert torch.equal(kp, want_k) and torch.equal(vp, want_v)


@pytest.mark.parametrize("nh,nkv,hd", [(8, 4, 256), (5, 1, 128), (18, 1, 64)])
def test_attn_decode_takes_partial_results_at_any_float(K, nh, nkv, hd):
    """Shares of a row that meet in memory: buffers that begin at a multiple of four bytes and not of sixteen give the same bits, from
    raw projections and from queries ready for use."""
    from agave_amd.ops import attention_mfma as A
    g = torch.Generator().manual_seed(hd)
    lens, n_pages = [700, 33], 13
    kp = torch.randn(n_pages, nkv, 64, hd, generator=g).bfloat16().to(DEV)
    vp = torch.randn(n_pages, nkv, hd, 64, generator=g).bfloat16().to(DEV)
    table = torch.tensor([list(range(11)), [11] + [-1] * 10], dtype=torch.int32, device=DEV)
    q = torch.randn(2, nh * hd, generator=g).bfloat16().to(DEV)
    made = []
    for off in (0, 1):
        step, asked = _FakeStep(lens, lambda L: L - 1, None), []
        real = step.workspace

        class Shifted:
            def get(self, name, rows, cols, dtype):
                asked.append(name)
                return real.get(name, rows * cols + 1, 1, dtype).view(-1)[off:off + rows * cols].view(rows, cols)
        step.workspace = Shifted()
        outs = [torch.full((2, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        A.decode_fused(q, None, None, outs[0], None, None, 0.0, 0.0, None, 1.0, kp, vp, table, _i32([0, 0]), step, nh, nkv, hd, 0.1, None)
        A.attention(q, outs[1], kp, vp, table, _i32([0, 0]), step, nh, nkv, hd, 0.1, None)
        assert asked.count("attn_part_o") == 2                 # (both in shares)
        made.append(outs)
    assert torch.isfinite(made[0][0].float()).all()
    for a, b in zip(*made):
        assert torch.equal(a, b)


@pytest.mark.parametrize("slices", [1, 2, 3, 4])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 4, 256), (5, 1, 128), (18, 1, 64)])
def test_attn_decode_fused_adds_slices_of_the_projections(K, nh, nkv, hd, slices):
    """Raw projections as 32-bit slices leave the bits that their sum leaves in bfloat16 (whole 64ths below 2: every sum is exact in
    both types).  The slices lie side by side, q, k and v of one product."""
    from agave_amd.ops import attention_mfma as A
    g = torch.Generator().manual_seed(slices)
    lens, cols = [1, 40, 64, 200, 97], (nh + 2 * nkv) * hd
    B, n_pages = len(lens), 12
    table = torch.full((B, 4), -1, dtype=torch.int32)
    perm = torch.randperm(n_pages, generator=g).tolist()
    for b, L in enumerate(lens):
        for i in range((L + 63) // 64):
            table[b, i] = perm.pop()
    parts = torch.randint(-31, 32, (slices, B, cols), generator=g).float() / 64
    whole = parts.sum(0).bfloat16()
    assert torch.equal(whole.float(), parts.sum(0))
    gain = (1 + 0.2 * torch.randn(hd, generator=g)).to(DEV)
    inv_freq = torch.exp(-torch.arange(hd // 2).float() / hd * 5).to(DEV)
    pages = [torch.randn(n_pages, nkv, 64, hd, generator=g).bfloat16().to(DEV), torch.randn(n_pages, nkv, hd, 64, generator=g).bfloat16().to(DEV)]
    step = _FakeStep(lens, lambda L: L - 1, None)
    outs = []
    for rows in (whole.to(DEV), parts.to(DEV)):
        q, k, v = rows.split((nh * hd, nkv * hd, nkv * hd), dim=-1)
        kp, vp = pages[0].clone(), pages[1].clone()
        out = torch.full((B, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        A.decode_fused(q, k, v, out, gain, gain, 1e-6, 1e-6, inv_freq, 1.0, kp, vp, table.to(DEV), _i32([0] * B), step, nh, nkv, hd, 0.1, None)
        outs.append((out, kp, vp))
    assert torch.isfinite(outs[0][0].float()).all()
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    # the q/k kernel of steps with several tokens a sequence, the same rows as a prompt's of one sequence
    pos, tab = _i32(list(range(60, 60 + B))), torch.tensor([[3, 1, -1, -1]], dtype=torch.int32).to(DEV)
    outs = []
    for rows in (whole.to(DEV), parts.to(DEV)):
        q, k, v = rows.split((nh * hd, nkv * hd, nkv * hd), dim=-1)
        kp, vp, q_rot = pages[0].clone(), pages[1].clone(), torch.full((B, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        K.qk_norm_rope_kv(q, k, v, q_rot, gain, gain, 1e-6, 1e-6, inv_freq, 1.0, _i32([0] * B), pos, kp, vp, tab, _i32([0]), nh, nkv, hd, packed=True)
        outs.append((q_rot, kp, vp))
    assert torch.isfinite(outs[0][0].float()).all()
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    q5 = torch.zeros(5, B, nh * hd, device=DEV)
    with pytest.raises(ValueError):
        A.decode_fused(q5, None, None, outs[0][0], gain, gain, 1e-6, 1e-6, inv_freq, 1.0, kp, vp, table.to(DEV), _i32([0] * B), step, nh, nkv,
                       hd, 0.1, None)
    with pytest.raises(ValueError):
        K.qk_norm_rope_kv(q5, None, None, outs[0][0], gain, None, 1e-6, 0.0, inv_freq, 1.0, _i32([0] * B), pos, None, None, None, None, nh, 0, hd)


# Heads as long as the kernel's tiles: a page's keys and values are asked for at once, one token's before its queries are there.
@pytest.mark.parametrize("nh,nkv,hd,window", [(8, 4, 64, 66), (34, 2, 64, None), (16, 4, 128, 130), (6, 6, 256, None), (4, 2, 256, 3)])
def test_attn_plain_heads_of_whole_tiles(K, nh, nkv, hd, window):
    for dtype in (torch.float32, torch.bfloat16):
        test_attn_plain_rows(K, dtype, nh, nkv, hd, window)
    if window is None:
        for n in (90, 170):
            test_attn_plain_values_that_are_not_finite(K, n, hd)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,n", [(8, 4, 256, 803), (6, 6, 256, 1011), (8, 4, 128, 1050)])
def test_attn_plain_long_heads_of_many_workgroups(K, dtype, nh, nkv, hd, n):
    """Heads of 256 (and of 128 in bfloat16), a page's keys at once (few workgroups) and one after another (many): a prompt's first rows
    are bit for bit the same whether the rest comes with them, and a token a sequence those of the same tokens among others."""
    few = 160
    g = torch.Generator().manual_seed(nh)
    pages = (n + 63) // 64
    kp, vp = (torch.randn(pages, nkv, *shape, generator=g).to(dtype).to(DEV) for shape in ((64, hd), (hd, 64)))
    q = torch.randn(n, nh * hd, generator=g).to(dtype).to(DEV)
    table = torch.randperm(pages, generator=g).to(torch.int32)[None].to(DEV)
    outs = []
    for m in (few, n):
        out = torch.full((m, nh * hd), float("nan"), dtype=dtype, device=DEV)
        K.attn_plain(q[:m], out, kp, vp, table, _i32([0]), _i32([0] * m), _i32(list(range(m))), nh, nkv, hd, 0.05, None)
        outs.append(out)
    assert torch.equal(outs[0], outs[1][:few]) and torch.isfinite(outs[1].float()).all()
    seqs, pos = 150, _i32([(37 * i) % (64 * pages) for i in range(150)])
    rows = []
    for m in (30, seqs):
        out = torch.empty(m, nh * hd, dtype=dtype, device=DEV)
        K.attn_plain(q[:m], out, kp, vp, table.expand(m, -1).contiguous(), _i32([0] * m), _i32(list(range(m))), pos[:m], nh, nkv, hd, 0.05, None,
                     one_token_each=True)
        rows.append(out)
    assert torch.equal(rows[0], rows[1][:30])
    k, v = kp.cpu().double()[table[0].cpu().long()], vp.cpu().double()[table[0].cpu().long()]
    k, v = k.permute(1, 0, 2, 3).reshape(nkv, -1, hd), v.permute(1, 0, 3, 2).reshape(nkv, -1, hd)
    tol = dict(atol=3e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    for got, t, p in ((outs[1], n - 1, n - 1), (outs[1], 200, 200), (rows[1], 149, int(pos[149]))):
        for h in range(nh):
            w = torch.softmax(0.05 * k[h * nkv // nh, :p + 1] @ q[t].cpu().double().view(nh, hd)[h], 0)
            assert torch.allclose(got[t].cpu().double().view(nh, hd)[h], w @ v[h * nkv // nh, :p + 1], **tol)


@pytest.mark.parametrize("hd", [64, 128, 256, 100])
def test_attn_plain_pages_that_are_not_there(K, hd):
    """Keys of pages that the table does not name count as unseen, the first, the last and one between, whoever asks for them first."""
    from agave_amd.parts import Workspace
    nh, nkv, ctx = 4, 2, 300
    g = torch.Generator().manual_seed(hd)
    kp, vp = (torch.randn(5, nkv, *shape, generator=g).to(DEV) for shape in ((64, hd), (hd, 64)))
    q = torch.randn(3, nh * hd, generator=g).to(DEV)
    table = torch.tensor([[-1, 1, 2, 3, 4], [0, 1, 9, 3, 4], [0, 1, 2, 3, -1]], dtype=torch.int32, device=DEV)
    k, v = kp.cpu().double(), vp.cpu().double()
    ref = torch.empty(3, nh, hd, dtype=torch.float64)
    for b, gone in enumerate((0, 2, 4)):
        seen = [i for i in range(ctx) if i // 64 != gone]
        for h in range(nh):
            keys = torch.stack([k[i // 64, h // 2, i % 64] for i in seen])
            vals = torch.stack([v[i // 64, h // 2, :, i % 64] for i in seen])
            ref[b, h] = torch.softmax(0.2 * keys @ q.cpu().double().view(3, nh, hd)[b, h], 0) @ vals
    for more in ({}, {"span": 5, "workspace": Workspace(torch.device(DEV))}):
        out = torch.empty_like(q)
        K.attn_plain(q, out, kp, vp, table, _i32([0] * 3), _i32([0, 1, 2]), _i32([ctx - 1] * 3), nh, nkv, hd, 0.2, None, one_token_each=True, **more)
        assert torch.allclose(out.cpu().double().view(3, nh, hd), ref, atol=2e-6 + 1e-7 * hd, rtol=2e-5)
