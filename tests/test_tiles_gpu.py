"""K's step 1 on pair tiles against the pair-map path and a plain FP64 sum,
at the sizes where it can go wrong: AO counts off the 16-row groups, aux rows
off the blocks of 8, occupied counts at the edges of the tile widths, AOs with
no stored pair, one and two factors, one storage or arithmetic type at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pair_list(rng, nao, fill, empty=()):
    """A screened pair list: each pair with probability ``fill`` (rows of
    their own densities), none for the AOs in ``empty``."""
    rows, cols = np.tril_indices(nao)
    p = np.clip(fill * (.2 + 1.6 * rng.random(nao)), 0, 1)
    keep = rng.random(len(rows)) < np.sqrt(p[rows] * p[cols])
    for i in empty:
        keep &= (rows != i) & (cols != i)
    return rows[keep], cols[keep]


def exact_k(cderi, rows, cols, nao, fl, fr):
    import torch
    a = torch.zeros((len(cderi), nao, nao), dtype=torch.float64, device='cuda')
    a[:, rows, cols] = cderi.double()
    a[:, cols, rows] = cderi.double()
    rl = (a.reshape(-1, nao) @ fl).reshape(len(cderi), nao, -1).transpose(0, 1).reshape(nao, -1)
    rr = rl if fr is None else (a.reshape(-1, nao) @ fr).reshape(len(cderi), nao, -1).transpose(0, 1).reshape(nao, -1)
    return rl @ rr.T.contiguous()


def inputs(nao, naux, nocc, two, storage='float64', seed=0, empty=()):
    import torch
    rng = np.random.default_rng(seed + 7 * nao + naux + 31 * nocc)
    rows, cols = pair_list(rng, nao, .4, empty)
    dt = getattr(torch, storage)
    cderi = torch.from_numpy(rng.standard_normal((naux, len(rows)))).cuda().to(dt)
    f = [torch.from_numpy(rng.standard_normal((nao, nocc))).cuda() for _ in range(1 + two)]
    addr = torch.from_numpy((rows * nao + cols).astype(np.int32)).cuda()
    return cderi, torch.from_numpy(rows).cuda(), torch.from_numpy(cols).cuda(), addr, f[0], f[1] if two else None


def make_tiles(addr, nao, lower=0, order_of=None):
    import torch
    from electrolites_amd import _dev, _lib
    pmap = torch.empty(nao * nao, dtype=torch.int32, device='cuda')
    _lib.call('mdf_build_pair_map', _dev.ptr(addr), len(addr), nao, _dev.ptr(pmap), _dev.stream_ptr())
    nb = _lib.query('mdf_pair_tiles_bytes', nao)
    buf = torch.full((nb,), 0x5a, dtype=torch.uint8, device='cuda')
    _lib.call('mdf_build_pair_tiles', _dev.ptr(pmap), nao, lower, _dev.ptr(order_of), _dev.ptr(buf), nb,
              _dev.stream_ptr())
    return pmap, buf


def get_k(cderi, pmap, tiles, nao, fl, fr, prec, rows=0):
    import torch
    from electrolites_amd import _dev, _lib, fastdf
    naux, npairs = cderi.shape
    nocc = fl.shape[1]
    q = 'mdf_get_k_workspace' if tiles is None else 'mdf_get_k_tiles_workspace'
    nb = _lib.query(q, naux, nao, nocc, int(fr is not None), prec, rows)
    # NaN workspace: every value that is used has to have been written
    work = torch.full((nb // 8 + 1,), float('nan'), dtype=torch.float64, device='cuda')
    vk = torch.full((nao, nao), float('nan'), dtype=torch.float64, device='cuda')
    _lib.call('mdf_get_k_tiles', _dev.ptr(cderi), fastdf._dtype_code(cderi), naux, npairs, cderi.stride(0),
              _dev.ptr(pmap), _dev.ptr(tiles), nao, _dev.ptr(fl), _dev.ptr(fr), nocc, nocc, prec, _dev.ptr(vk), nao,
              0, _dev.ptr(work), nb, _dev.stream_ptr())
    return vk


def rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize('nao,naux,nocc', [
    (1, 1, 1), (16, 8, 16), (17, 9, 17), (31, 7, 63), (33, 15, 64), (112, 16, 65), (129, 17, 129), (130, 3, 161),
    (145, 8, 193), (131, 5, 257), (128, 2, 321)])
@pytest.mark.parametrize('two', [False, True])
def test_k_tiles_fp64(nao, naux, nocc, two):
    print(f'k tiles nao {nao} naux {naux} nocc {nocc} two {two}', flush=True)
    empty = (0, nao - 1, nao // 2) if nao > 16 else ()
    cderi, rows, cols, addr, fl, fr = inputs(nao, naux, nocc, two, empty=empty)
    if not len(addr):
        pytest.skip('no pair drawn')
    pmap, buf = make_tiles(addr, nao)
    vk = get_k(cderi, pmap, buf, nao, fl, fr, 0)
    # a product of n terms in any order is within n eps of the exact one
    tol = 2.3e-16 * (nao + naux * nocc)
    assert rel(vk, exact_k(cderi, rows, cols, nao, fl, fr)) < tol
    assert rel(vk, get_k(cderi, pmap, None, nao, fl, fr, 0)) < 2 * tol


@pytest.mark.parametrize('storage,prec', [('float32', 0), ('float32', 1), ('float64', 1)])
@pytest.mark.parametrize('nao,naux,nocc', [(33, 9, 17), (130, 12, 161), (150, 5, 320)])
def test_k_tiles_types(storage, prec, nao, naux, nocc):
    print(f'k tiles {storage} prec {prec} nao {nao} naux {naux} nocc {nocc}', flush=True)
    cderi, rows, cols, addr, fl, _ = inputs(nao, naux, nocc, False, storage)
    pmap, buf = make_tiles(addr, nao)
    vk = get_k(cderi, pmap, buf, nao, fl, None, prec)
    tol = (2.3e-16 if prec == 0 else 1.2e-7) * (nao + naux * nocc) ** (1 if prec == 0 else .5)
    assert rel(vk, exact_k(cderi, rows, cols, nao, fl, None)) < tol


@pytest.mark.parametrize('storage', ['float32', 'float64'])
@pytest.mark.parametrize('two', [False, True])
@pytest.mark.parametrize('nao,naux,nocc', [(33, 9, 17), (64, 8, 128), (130, 12, 161), (97, 7, 256), (150, 5, 320)])
def test_k_tiles_split_bf16(storage, two, nao, naux, nocc):
    print(f'k tiles bf16x3 {storage} two {two} nao {nao} naux {naux} nocc {nocc}', flush=True)
    cderi, rows, cols, addr, fl, fr = inputs(nao, naux, nocc, two, storage)
    pmap, buf = make_tiles(addr, nao)
    ref = exact_k(cderi, rows, cols, nao, fl, fr)
    vk = get_k(cderi, pmap, buf, nao, fl, fr, 2)
    # hi + lo holds 2^-17 of a value and the dropped lo lo term is below
    # 2^-16 of a product, in each of two steps
    assert rel(vk, ref) < 4 * 2. ** -16
    assert rel(vk, ref) < 1.2 * rel(get_k(cderi, pmap, None, nao, fl, fr, 2), ref) + 1e-7


def test_k_tiles_passes():
    """Passes of fewer aux rows than a block of 8, and of several blocks."""
    cderi, rows, cols, addr, fl, _ = inputs(60, 37, 20, False)
    pmap, buf = make_tiles(addr, 60)
    ref = exact_k(cderi, rows, cols, 60, fl, None)
    for nrow in (1, 5, 8, 13):
        print(f'k tiles passes of {nrow}', flush=True)
        assert rel(get_k(cderi, pmap, buf, 60, fl, None, 0, nrow), ref) < 2.3e-16 * (60 + 37 * 20)


@pytest.mark.parametrize('nao', [5, 16, 47, 130, 600, 2060])
def test_tiles_hold_every_pair_once(nao):
    """Rows are a permutation; the map holds each stored pair in both orders,
    and its lower half each off-group pair once and each in-group pair twice
    with the factor 1/2."""
    import torch
    print(f'tiles nao {nao}', flush=True)
    rng = np.random.default_rng(nao)
    rows, cols = pair_list(rng, nao, .1 if nao > 500 else .4, (nao // 3,))
    addr = torch.from_numpy((rows * nao + cols).astype(np.int32)).cuda()
    _, buf = make_tiles(addr, nao)
    _, low = make_tiles(addr, nao, 1, buf)
    G, C = (nao + 15) // 16, (nao + 31) // 32 * 32 + 32
    half = 1 << 30
    for which, b in (('full', buf), ('lower', low)):
        w = b.cpu().numpy()[:(len(b) // 4) * 4].view(np.int32)
        r = w[:16 * G].reshape(G, 16)
        nstep = w[16 * G:17 * G]
        o = (17 * G + 63) // 64 * 64
        cc = w[o:o + G * C].reshape(G, C)
        o = (o + G * C + 63) // 64 * 64
        m = w[o:o + G * C * 16].reshape(G, C // 16, 16, 16)
        assert sorted(r[r >= 0]) == list(range(nao)) and np.all(r.reshape(-1)[nao:] == -1)
        got = np.zeros((nao, nao))
        for g in range(G):
            n = nstep[g] * 16
            c = cc[g]
            real = c[c < nao]
            assert np.all(c[len(real):] == nao) and np.all(np.diff(real) > 0) and n == -(-len(real) // 16) * 16
            mm = m[g].transpose(1, 0, 2).reshape(16, C)
            assert np.all(mm[:, len(real):] == -1)
            ii, kk = np.nonzero(mm >= 0)
            e = mm[ii, kk]
            i, j = r[g][ii], c[kk]
            p = e & (half - 1)
            assert np.all(rows[p] == np.maximum(i, j)) and np.all(cols[p] == np.minimum(i, j))
            np.add.at(got, (i, j), np.where(e & half, .5, 1.))
        want = np.zeros((nao, nao))
        want[rows, cols] = want[cols, rows] = 1.
        if which == 'lower':
            got = got + got.T
        assert np.array_equal(got, want)


@pytest.mark.parametrize('storage', ['float64', 'float32'])
@pytest.mark.parametrize('lower', [0, 1])
@pytest.mark.parametrize('nao,nL,nocc', [(17, 9, 5), (47, 8, 33), (130, 11, 97), (150, 3, 321)])
def test_step1_tiles(storage, lower, nao, nL, nocc):
    """R = A F, and R = T F with T + T^T = A: F^T T F + its transpose."""
    import torch
    from electrolites_amd import _dev, _lib, fastdf
    print(f'step1 tiles {storage} lower {lower} nao {nao} nL {nL} nocc {nocc}', flush=True)
    cderi, rows, cols, addr, f, _ = inputs(nao, nL, nocc, False, storage, empty=(1,))
    _, buf = make_tiles(addr, nao, lower)
    nb = _lib.query('mdf_k_step1_tiles_workspace', nao, nocc)
    work = torch.full((nb // 8,), float('nan'), dtype=torch.float64, device='cuda')
    ldr = nocc + 3
    R = torch.full((nL, nao, ldr), float('nan'), dtype=torch.float64, device='cuda')
    _lib.call('mdf_k_step1_tiles', _dev.ptr(cderi), fastdf._dtype_code(cderi), nL, len(addr), cderi.stride(0),
              _dev.ptr(buf), lower, nao, _dev.ptr(f), nocc, nocc, _dev.ptr(R), ldr, nao * ldr, _dev.ptr(work), nb,
              _dev.stream_ptr())
    a = torch.zeros((nL, nao, nao), dtype=torch.float64, device='cuda')
    a[:, rows, cols] = cderi.double()
    a[:, cols, rows] = cderi.double()
    got, want = R[:, :, :nocc], a @ f
    assert bool(R[:, :, nocc:].isnan().all())
    if lower:
        got = f.T @ got
        got, want = got + got.transpose(1, 2), f.T @ want
    assert rel(got, want) < 2.3e-16 * 4 * nao


@pytest.mark.parametrize('nao,nocc,batch', [(16, 1, 1), (33, 5, 8), (120, 16, 9), (203, 17, 3), (300, 50, 17)])
@pytest.mark.parametrize('init', [False, True])
def test_gemm_pairs_tiles(nao, nocc, batch, init):
    """A symmetric product's values at the stored pairs, from the lower tiles
    and from the general entry (which reads its own lower triangle), against
    a plain sum; every other entry of W keeps its value.  Two AOs have no
    pair; the rows of W and of the factors are padded."""
    import ctypes
    import torch
    from electrolites_amd import _dev, _lib
    rng = np.random.default_rng(nao + nocc + batch)
    rows, cols = pair_list(rng, nao, .4, (0, nao - 1))
    npairs = len(rows)
    addr = torch.from_numpy((rows * nao + cols).astype(np.int32)).cuda()
    _, tiles = make_tiles(addr, nao, 1)
    f = torch.zeros((nao, nocc + 3), dtype=torch.float64, device='cuda')
    f[:, :nocc] = torch.from_numpy(rng.standard_normal((nao, nocc))).cuda()
    m = torch.from_numpy(rng.standard_normal((batch, nocc, nocc))).cuda()
    m = m + m.transpose(1, 2)
    h = torch.zeros((nao, batch * nocc + 1), dtype=torch.float64, device='cuda')
    h[:, :batch * nocc] = torch.matmul(f[:, :nocc], m).transpose(0, 1).reshape(nao, -1)
    w = torch.from_numpy(rng.standard_normal((batch, npairs + 5))).cuda()
    sc, vals = (torch.from_numpy(rng.standard_normal(n)).cuda() for n in (batch, npairs))
    p = torch.matmul(torch.matmul(f[:, :nocc], m), f[:, :nocc].T)
    r, c = torch.from_numpy(rows).cuda(), torch.from_numpy(cols).cuda()
    base = sc[:, None] * vals if init else w[:, :npairs]
    base = base.clone()
    ref = torch.cat([base - .6 * p[:, r, c], w[:, npairs:]], dim=1)
    if init:
        w[:, :npairs] = float('nan')
    g = w.clone()
    isc = (_dev.ptr(sc), _dev.ptr(vals)) if init else (None, None)
    _lib.call('mdf_gemm_pairs_tiles', nao, nocc, ctypes.c_double(-.6), _dev.ptr(f), nocc + 3, _dev.ptr(h),
              h.shape[1], nocc, _dev.ptr(tiles), npairs, _dev.ptr(w), npairs + 5, *isc, batch, _dev.stream_ptr())
    cmap = torch.full((nao * (nao + 1) // 2,), -1, dtype=torch.int32, device='cuda')
    cmap[r * (r + 1) // 2 + c] = torch.arange(npairs, dtype=torch.int32, device='cuda')
    _lib.call('mdf_gemm_pairs_batched', 1, nao, nocc, ctypes.c_double(-.6), _dev.ptr(f), nocc + 3, 0, _dev.ptr(h),
              h.shape[1], nocc, _dev.ptr(cmap), _dev.ptr(g), npairs + 5, *isc, batch, _dev.stream_ptr())
    # two products of nocc terms each, both sides rounding every one:
    # 4 nocc eps sum |f| |m| |f|, and the sum with the base
    bound = 4 * 2.3e-16 * (nocc * float(f.abs().max()) ** 2 * float(m.abs().sum(dim=(1, 2)).max()) +
                           float(base.abs().max()))
    assert float((w - ref).abs().max()) < bound
    assert float((w - g).abs().max()) < bound


@pytest.mark.parametrize('built', [False, True])
def test_captured_call(built):
    """get_jk of response densities (no value goes to the host) captured with
    the tiles not built yet, or built: each replay, with eager calls between,
    gives the eager result, and the eager calls stay right afterwards."""
    import torch
    from electrolites_amd import fastdf
    nao, naux, nocc = 150, 40, 20
    cderi, rows, cols, addr, fl, fr = inputs(nao, naux, nocc, True)
    print(f'captured get_jk, tiles built {built}', flush=True)

    class DF:
        def __init__(self):
            self._cderi, self._cderi_idx = {0: cderi}, (addr, None)
    x = fl @ (2. * fr).T
    dm = fastdf.tag_array(x + x.T, mo1=fl, occ_coeff=fr, symmetrize=1)
    refs = [t.clone() for t in fastdf.get_jk(DF(), dm, hermi=1)]     # sizes the shared workspace
    df = DF()
    fastdf.get_jk(df, dm, hermi=1, with_k=built)
    assert bool(df._mdf_layout[2]._tiles) == built
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        vj, vk = fastdf.get_jk(df, dm, hermi=1)
    for rep in range(3):
        vj.zero_()
        vk.zero_()
        eager = fastdf.get_jk(df, dm, hermi=1)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for got in ((vj, vk), eager):
            assert torch.equal(got[0], refs[0])
            assert rel(got[1], refs[1]) < 2.3e-16 * 2 * (nao + naux * nocc)


@pytest.mark.parametrize('tiled', [False, True])
@pytest.mark.parametrize('two', [False, True])
@pytest.mark.parametrize('nocc', [(1 << 22) - 3, (1 << 22) + 5])
def test_k_rows_beyond_32_bits(monkeypatch, tiled, two, nocc):
    """The transformed blocks of 130 functions and 2^22 columns span more
    than 2^32 values (step 2's row offsets); a factor of more columns than
    one contraction takes is summed in parts."""
    import torch
    monkeypatch.setenv('MDF_K_BLOCK_BYTES', str(80 << 30))
    nao, naux = 130, 8
    print(f'k rows nao {nao} nocc {nocc} tiled {tiled} two {two}', flush=True)
    cderi, rows, cols, addr, _, _ = inputs(nao, naux, 1, False)
    pmap, buf = make_tiles(addr, nao)
    g = torch.Generator(device='cuda').manual_seed(nocc)
    fl = torch.randn((nao, nocc), generator=g, dtype=torch.float64, device='cuda')
    fr = torch.randn((nao, nocc), generator=g, dtype=torch.float64, device='cuda') if two else None
    vk = get_k(cderi, pmap, buf if tiled else None, nao, fl, fr, 0)
    a = torch.zeros((naux, nao, nao), dtype=torch.float64, device='cuda')
    a[:, rows, cols] = cderi
    a[:, cols, rows] = cderi
    m = fl @ (fl if fr is None else fr).T
    ref = sum(x @ m @ x for x in a)
    # naux nocc products a sum in any order; random signs, so their number
    # counts by its root
    assert rel(vk, ref) < 2.3e-16 * 4 * (naux * nocc) ** .5


@pytest.mark.parametrize('prec', [0, 1])
@pytest.mark.parametrize('two', [False, True])
@pytest.mark.parametrize('nocc', [1, 3, 5, 18])
def test_k_short_blocks(prec, two, nocc):
    """Passes of one block of fewer than 8 aux rows, the last pass shorter
    still, with rows of every remainder by the 16-byte pieces."""
    nao, naux = 37, 17
    cderi, rows, cols, addr, fl, fr = inputs(nao, naux, nocc, two)
    pmap, buf = make_tiles(addr, nao)
    ref = exact_k(cderi, rows, cols, nao, fl, fr)
    tol = 2.3e-16 * (nao + naux * nocc) if prec == 0 else 1.2e-7 * (nao + naux * nocc) ** .5
    for nrow in (1, 2, 3, 5, 7, 8, 9):
        for tiles in (None, buf):
            print(f'k short blocks prec {prec} two {two} nocc {nocc} rows {nrow} tiled {tiles is not None}', flush=True)
            assert rel(get_k(cderi, pmap, tiles, nao, fl, fr, prec, nrow), ref) < tol


@pytest.mark.parametrize('prec', [0, 1, 2])
@pytest.mark.parametrize('two', [False, True])
def test_one_function(prec, two):
    """nao 1: one pair, one group of one row and one column."""
    import torch
    print(f'one function prec {prec} two {two}', flush=True)
    rng = np.random.default_rng(prec)
    cderi = torch.from_numpy(rng.standard_normal((9, 1))).cuda()
    addr = torch.zeros(1, dtype=torch.int32, device='cuda')
    fl, fr = (torch.from_numpy(rng.standard_normal((1, 3))).cuda() for _ in range(2))
    pmap, buf = make_tiles(addr, 1)
    got = get_k(cderi, pmap, buf, 1, fl, fr if two else None, prec)
    ref = (cderi ** 2).sum() * (fl * (fr if two else fl)).sum()
    assert float((got - ref).abs()) < (1e-14, 1e-5, 1e-3)[prec] * float((cderi ** 2).sum() * (fl * fl).sum().sqrt() *
                                                                        (fr * fr + fl * fl).sum().sqrt())


def test_tiles_of_many_functions():
    """The row order's widest form (from 8193 functions on): a permutation
    of the rows, and in the map each pair once, at its row and column."""
    import torch
    nao = 8250
    print(f'tiles nao {nao}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(1)
    near = torch.randint(0, nao, (nao, 12), generator=g, device='cuda')
    rows = torch.arange(nao, device='cuda').repeat_interleave(12)
    near = near.reshape(-1)
    pair = torch.unique(torch.cat([torch.maximum(rows, near) * nao + torch.minimum(rows, near),
                                   torch.arange(nao, device='cuda') * (nao + 1)]))
    _, buf = make_tiles(pair.to(torch.int32), nao)
    w = buf[:buf.numel() // 4 * 4].view(torch.int32)
    G, C = (nao + 15) // 16, (nao + 31) // 32 * 32 + 32
    r = w[:16 * G]
    assert torch.equal(torch.sort(r[:nao])[0], torch.arange(nao, dtype=torch.int32, device='cuda'))
    assert bool((r[nao:] == -1).all())
    o = (17 * G + 63) // 64 * 64
    cols = w[o:o + G * C].reshape(G, C)
    o = (o + G * C + 63) // 64 * 64
    m = w[o:o + G * C * 16].reshape(G, C // 16, 16, 16).transpose(1, 2).reshape(G, 16, C)
    gi, ii, kk = torch.nonzero(m >= 0, as_tuple=True)
    i, j, p = r.reshape(G, 16)[gi, ii].long(), cols[gi, kk].long(), m[gi, ii, kk].long()
    assert torch.equal(pair[p], torch.maximum(i, j) * nao + torch.minimum(i, j))
    # every off-diagonal pair in both orders
    assert torch.unique(i * nao + j).numel() == i.numel() == 2 * pair.numel() - nao


def test_layout_tiles_on_another_stream():
    """Tiles built on one stream behind queued work, used by a call on
    another: the single-stream result."""
    import torch
    from electrolites_amd import fastdf
    nao, naux, nocc = 150, 40, 20
    cderi, rows, cols, addr, f, _ = inputs(nao, naux, nocc, False)
    print('layout tiles on another stream', flush=True)

    class DF:
        def __init__(self):
            self._cderi, self._cderi_idx = {0: cderi}, (addr, None)
    dm = fastdf.tag_array(f @ f.T, mo_coeff=f, mo_occ=torch.ones(nocc, dtype=torch.float64, device='cuda'))
    ref = fastdf.get_jk(DF(), dm, hermi=1)[1].clone()
    df = DF()
    lay = fastdf._layout(df, cderi, nao)
    big = torch.randn(4096, 4096, device='cuda', dtype=torch.float64)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        for _ in range(4):
            big @ big
        assert lay.tiles() is not None
    with torch.cuda.stream(b):
        vk = fastdf.get_jk(df, dm, hermi=1)[1]
    torch.cuda.synchronize()
    assert torch.equal(vk, ref)
