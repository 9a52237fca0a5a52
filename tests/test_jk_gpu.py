"""GPU parity of the HIP J/K path against the FP64 oracle.

Follows the reference's DF suite (tests/test_df.py:78-135): several
molecules, hermi 0/1, mo-tagged and plain densities, n_dm 1/2/4/5, and the
bar max|got - ref| / max|ref| <= 1e-12 (the reference's own bar is 1e-11,
tests/test_df.py:40; the target here is 1e-12).
"""
import numpy as np
import pytest

from oracle import oracle as O

TOL = 1e-12


def rel(a, b):
    return np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(b).max(), 1e-300)


class FakeDF:
    """A DF object carrying a given cderi (the reference's DF fields)."""

    def __init__(self, cderi, pair_addr, nao):
        import torch
        self._cderi = {0: torch.from_numpy(np.ascontiguousarray(cderi)).cuda()}
        rows, cols = np.divmod(pair_addr, nao)
        self._cderi_idx = (pair_addr.astype(np.int32), np.where(rows == cols)[0])

    def build(self):
        raise AssertionError('cderi given')


@pytest.fixture(scope='module')
def water2():
    from electrolites_amd.gto import water_cluster
    mol = water_cluster(2, seed=1, side=4.0)
    ao, aux = mol.ao.as_dict(), mol.aux.as_dict()
    j3c = O.int3c2e(ao, aux)
    j2c = O.int2c2e(aux)
    pa, _ = O.pair_addresses(mol.nao)
    cderi = O.cholesky_eri(j3c, j2c, pa)
    return mol.nao, cderi, pa


def rand_psd(nao, nocc, rng):
    c = np.linalg.qr(rng.standard_normal((nao, nocc)))[0]
    return c


@pytest.mark.gpu
@pytest.mark.parametrize('tagged', [True, False])
def test_water_dimer_jk(water2, tagged):
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    rng = np.random.default_rng(20260917)
    c = rand_psd(nao, 10, rng)
    dm = 2 * c @ c.T
    if tagged:
        dm = fastdf.tag_array(dm, mo_coeff=c, mo_occ=np.full(10, 2.))
    df = FakeDF(cderi, pa, nao)
    vj, vk = fastdf.get_jk(df, dm, hermi=1)
    rj, rk = O.get_jk(cderi, pa, np.asarray(dm))
    assert rel(vj, rj) < TOL
    assert rel(vk, rk) < TOL
    assert isinstance(vj, np.ndarray) and vj.shape == (nao, nao)


@pytest.mark.gpu
def test_hermi0_nonsymmetric(water2):
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    rng = np.random.default_rng(11)
    dm = rng.standard_normal((nao, nao)) * .1
    df = FakeDF(cderi, pa, nao)
    vj, vk = fastdf.get_jk(df, dm, hermi=0)
    rj = O.get_j(cderi, pa, dm, hermi=0)
    rk = O.get_k(cderi, pa, dm)
    assert rel(vj, rj) < TOL
    assert rel(vk, rk) < 1e-11          # through an SVD of a random matrix


@pytest.mark.gpu
@pytest.mark.parametrize('n_dm', [2, 5])
def test_many_densities(water2, n_dm):
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    rng = np.random.default_rng(12)
    dms = []
    for _ in range(n_dm):
        a = rng.standard_normal((nao, nao)) * 1e-3
        dms.append(a + a.T)
    dms = np.array(dms)
    df = FakeDF(cderi, pa, nao)
    vj, vk = fastdf.get_jk(df, dms, hermi=1)
    rj, rk = O.get_jk(cderi, pa, dms)
    assert vj.shape == dms.shape
    assert rel(vj, rj) < TOL
    assert rel(vk, rk) < 1e-11


@pytest.mark.gpu
def test_j_only_branch(water2):
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    rng = np.random.default_rng(3)
    c = rand_psd(nao, 9, rng)
    dm = 2 * c @ c.T
    df = FakeDF(cderi, pa, nao)
    vj, vk = fastdf.get_jk(df, dm, hermi=1, with_k=False)
    assert vk is None
    assert rel(vj, O.get_j(cderi, pa, dm)) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize('nao,naux,nocc', [(37, 19, 5), (64, 130, 17),
                                           (129, 300, 64), (200, 611, 90), (240, 300, 170)])
def test_synthetic_shapes(nao, naux, nocc):
    """Ragged shapes: odd npairs (scalar loads), tile tails, nocc not a
    multiple of the MFMA tile."""
    from electrolites_amd import fastdf
    rng = np.random.default_rng(nao * 1000 + naux)
    pa, _ = O.pair_addresses(nao)
    cderi = rng.standard_normal((naux, len(pa)))
    c = rand_psd(nao, nocc, rng)
    dm = fastdf.tag_array(2 * c @ c.T, mo_coeff=c, mo_occ=np.full(nocc, 2.))
    df = FakeDF(cderi, pa, nao)
    vj, vk = fastdf.get_jk(df, dm, hermi=1)
    rj = O.get_j(cderi, pa, np.asarray(dm))
    rk = O.get_k_factor(cderi, pa, c * np.sqrt(2.))
    assert rel(vj, rj) < TOL
    assert rel(vk, rk) < TOL


@pytest.mark.gpu
def test_screened_pairs():
    """A cderi over a subset of the pairs (screening), K through the pair
    map; dropped pairs act as zeros in the unpacked matrix."""
    from electrolites_amd import fastdf
    nao, naux, nocc = 90, 150, 12
    rng = np.random.default_rng(5)
    pa_full, _ = O.pair_addresses(nao)
    keep = rng.random(len(pa_full)) > .3
    rows, cols = np.divmod(pa_full, nao)
    keep |= rows == cols
    pa = pa_full[keep]
    cderi = rng.standard_normal((naux, len(pa)))
    c = rand_psd(nao, nocc, rng)
    dm = fastdf.tag_array(2 * c @ c.T, mo_coeff=c, mo_occ=np.full(nocc, 2.))
    df = FakeDF(cderi, pa, nao)
    vj, vk = fastdf.get_jk(df, dm, hermi=1)
    assert rel(vj, O.get_j(cderi, pa, np.asarray(dm))) < TOL
    assert rel(vk, O.get_k_factor(cderi, pa, c * np.sqrt(2.))) < TOL


@pytest.mark.gpu
def test_k_block_partition(water2, monkeypatch):
    """K over many small aux blocks equals one block (the reference's block
    partition test, tests/test_df.py:279-301)."""
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    rng = np.random.default_rng(7)
    c = rand_psd(nao, 10, rng)
    dm = fastdf.tag_array(2 * c @ c.T, mo_coeff=c, mo_occ=np.full(10, 2.))
    df = FakeDF(cderi, pa, nao)
    _, vk1 = fastdf.get_jk(df, dm, hermi=1)
    monkeypatch.setattr(fastdf, 'K_WORKSPACE_BYTES', nao * 10 * 8 * 7)
    _, vk2 = fastdf.get_jk(df, dm, hermi=1)
    assert rel(vk2, vk1) < 1e-14


@pytest.mark.gpu
def test_device_in_device_out(water2):
    import torch
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    rng = np.random.default_rng(8)
    c = rand_psd(nao, 10, rng)
    dm = torch.from_numpy(2 * c @ c.T).cuda()
    fastdf.tag_array(dm, mo_coeff=torch.from_numpy(c).cuda(),
                     mo_occ=torch.full((10,), 2., dtype=torch.float64).cuda())
    vj, vk = fastdf.get_jk(FakeDF(cderi, pa, nao), dm, hermi=1)
    assert vj.is_cuda and vk.is_cuda
    rj, rk = O.get_jk(cderi, pa, 2 * c @ c.T)
    assert rel(vj.cpu().numpy(), rj) < TOL and rel(vk.cpu().numpy(), rk) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('nao,naux,nocc,mode,screened', [(64, 130, 17, 0, False), (200, 611, 90, 0, False),
                                                         (200, 300, 45, 1, False), (170, 260, 33, 0, True),
                                                         (150, 200, 40, 1, True), (230, 280, 170, 0, False),
                                                         (200, 260, 161, 1, True)])
def test_low_precision_k_error(precision, nao, naux, nocc, mode, screened):
    """FP32 and split-BF16 exchange against the FP64 oracle: one factor
    (mo-tagged) and two factors (untagged), full and screened pair sets,
    shapes that reach every A-operand case (below, above and across the
    diagonal).  Bar: 1e-5 relative to max |K| (FP32-level rounding; the split
    keeps 16 significand bits per operand and three of the four products)."""
    from electrolites_amd import fastdf
    rng = np.random.default_rng(nao + 7 + 100 * mode)
    pa, _ = O.pair_addresses(nao)
    if screened:
        rows, cols = np.divmod(pa, nao)
        pa = pa[(rng.random(len(pa)) > .25) | (rows == cols)]
    cderi = rng.standard_normal((naux, len(pa))) * .1
    c = rand_psd(nao, nocc, rng)
    dm = 2 * c @ c.T
    if mode == 0:
        dm = fastdf.tag_array(dm, mo_coeff=c, mo_occ=np.full(nocc, 2.))
    df = FakeDF(cderi, pa, nao)
    df.k_precision = precision
    _, vk = fastdf.get_jk(df, dm, hermi=1)
    rk = O.get_k(cderi, pa, np.asarray(dm))
    err = rel(vk, rk)
    print(f'{precision} mode {mode} screened {screened}: K rel err {err:.2e}')
    assert 1e-12 < err < 1e-5, err


@pytest.mark.gpu
@pytest.mark.parametrize('mode,screened,n_dm', [(0, False, 1), (1, False, 3), (0, True, 2), (1, True, 1)])
def test_fp32_storage(mode, screened, n_dm):
    """FP32-stored cderi (the reference's FASTDF_FP32 mode): J and K equal the
    FP64 oracle on the FP32-rounded tensor widened to FP64 (1e-12 / 1e-11
    relative), for one and two factors, full and screened pair sets; the
    narrow K modes read it too (1e-5)."""
    import torch
    from electrolites_amd import fastdf
    nao, naux, nocc = 150, 310, 37
    rng = np.random.default_rng(50 + 10 * mode + n_dm)
    pa, _ = O.pair_addresses(nao)
    if screened:
        rows, cols = np.divmod(pa, nao)
        pa = pa[(rng.random(len(pa)) > .3) | (rows == cols)]
    cd32 = (rng.standard_normal((naux, len(pa))) * .1).astype(np.float32)
    cs = [rand_psd(nao, nocc, rng) for _ in range(n_dm)]
    dm = np.array([2 * c @ c.T for c in cs])
    if mode == 0:
        dm = fastdf.tag_array(dm, mo_coeff=np.array(cs), mo_occ=np.full((n_dm, nocc), 2.))
    df = FakeDF(cd32.astype(np.float64), pa, nao)
    df._cderi = {0: torch.from_numpy(cd32).cuda()}
    assert df._cderi[0].dtype == torch.float32
    vj, vk = fastdf.get_jk(df, dm, hermi=1)
    rj, rk = O.get_jk(cd32.astype(np.float64), pa, np.asarray(dm))
    assert rel(vj, rj) < 1e-12
    assert rel(vk, rk) < 1e-11
    for prec in ('fp32', 'bf16x3'):
        df.k_precision = prec
        _, vkl = fastdf.get_jk(df, dm, hermi=1)
        assert rel(vkl, rk) < 1e-5, prec


@pytest.mark.gpu
def test_uhf_shapes_and_zero_density(water2):
    """UHF-shaped inputs, as GPU4PySCF's UHF passes them: (2, nao, nao) tagged
    with per-spin mo_coeff / mo_occ (occupations 0/1, different electron
    counts per spin; only occupied columns form the factor), and untagged
    (2, 2, nao, nao) stacks; outputs keep the input shape.  A zero density
    (no occupied orbital) returns the inputs, as the reference does
    (fastdf.py:850-851)."""
    from electrolites_amd import fastdf
    nao, cderi, pa = water2
    df = FakeDF(cderi, pa, nao)
    rng = np.random.default_rng(21)
    nmo = nao
    C = np.array([np.linalg.qr(rng.standard_normal((nao, nmo)))[0] for _ in range(2)])
    occ = np.zeros((2, nmo))
    occ[0, :6] = 1.
    occ[1, :4] = 1.
    dm = np.array([(C[s] * occ[s]) @ C[s].T for s in range(2)])
    tagged = fastdf.tag_array(dm, mo_coeff=C, mo_occ=occ)
    vj, vk = fastdf.get_jk(df, tagged, hermi=1)
    assert vj.shape == vk.shape == (2, nao, nao)
    rj, rk = O.get_jk(cderi, pa, dm)
    assert rel(vj, rj) < 1e-12 and rel(vk, rk) < 1e-11
    d4 = np.array([dm, dm[::-1] * .5])                     # (2, 2, nao, nao)
    vj4, vk4 = fastdf.get_jk(df, d4, hermi=1)
    assert vj4.shape == vk4.shape == d4.shape
    rj4, rk4 = O.get_jk(cderi, pa, d4.reshape(-1, nao, nao))
    assert rel(vj4.reshape(-1, nao, nao), rj4) < 1e-12 and rel(vk4.reshape(-1, nao, nao), rk4) < 1e-11
    z = fastdf.tag_array(np.zeros((nao, nao)), mo_coeff=C[0], mo_occ=np.zeros(nmo))
    out = fastdf.get_jk(df, z, hermi=1)
    assert out[0] is z and out[1] is z


@pytest.mark.gpu
@pytest.mark.parametrize('chunk_bytes', [None, 150000])
def test_ri_j_without_cderi(chunk_bytes):
    """J from three-centre integrals contracted on the fly (the reference's
    fastdfj3c.get_j) equals J from the stored cderi and the oracle's J, for
    several densities, hermi 1 and 0, one chunk or many."""
    from electrolites_amd import fastdf, fastdfj3c
    from electrolites_amd.df import DF
    from electrolites_amd.gto import water_cluster
    mol = water_cluster(3, seed=8, side=5.5, li=True)
    df = DF(mol).build()
    rng = np.random.default_rng(9)
    nao = mol.nao
    a = rng.standard_normal((3, nao, nao)) * .1
    dms = a + a.transpose(0, 2, 1)
    dfj = DF(mol)
    fastdfj3c._state(dfj, chunk_bytes)
    if chunk_bytes:
        assert len(dfj._mdf_j3c.tasks) > 1
    vj = dfj.get_j(dms, hermi=1)
    rj, _ = fastdf.get_jk(df, dms, hermi=1, with_k=False)
    assert rel(vj, rj) < 1e-12
    oj, _ = O.get_jk(df.cderi().cpu().numpy(), df._cderi_idx[0], dms)
    assert rel(vj, oj) < 1e-11
    ns = rng.standard_normal((nao, nao)) * .1                # hermi 0 (non-symmetric)
    vj0 = dfj.get_j(ns, hermi=0)
    rj0, _ = fastdf.get_jk(df, ns, hermi=0, with_k=False)
    assert rel(vj0, rj0) < 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize('nocc', [1, 5, 9])
def test_fp32_step2_flush_length(nocc):
    """FP32 step 2 keeps at most the products of 32 K-steps of one aux row
    (32 nocc for nocc <= 16) in one FP32 sum: over positive values the error
    is that of such sums added in FP64, taken here on the CPU one product
    after the other, which rounds more often than the matrix instruction."""
    import torch
    from electrolites_amd import _dev, _lib
    nao, naux = 48, 120000
    rng = np.random.default_rng(nocc)
    a = (rng.random((naux, nao)) + .5).astype(np.float32)
    cderi = torch.from_numpy(a.astype(np.float64)).cuda()        # diagonal pairs only: R = a exactly
    addr = torch.arange(nao, dtype=torch.int32, device='cuda') * (nao + 1)
    pmap = torch.empty(nao * nao, dtype=torch.int32, device='cuda')
    _lib.call('mdf_build_pair_map', _dev.ptr(addr), nao, nao, _dev.ptr(pmap), _dev.stream_ptr())
    f = torch.ones((nao, nocc), dtype=torch.float64, device='cuda')
    vk = torch.empty((nao, nao), dtype=torch.float64, device='cuda')
    nb = _lib.query('mdf_get_k_workspace', naux, nao, nocc, 0, 1, 0)
    work = torch.empty(nb, dtype=torch.uint8, device='cuda')
    print(f'fp32 flush nocc {nocc}', flush=True)
    _lib.call('mdf_get_k', _dev.ptr(cderi), 0, naux, nao, nao, _dev.ptr(pmap), nao, _dev.ptr(f), None, nocc, nocc, 1,
              _dev.ptr(vk), nao, 0, _dev.ptr(work), nb, _dev.stream_ptr())
    low = np.tril_indices(nao)
    exact = nocc * (a.T.astype(np.float64) @ a.astype(np.float64))[low]
    p = (a[:, low[0]].astype(np.float64) * a[:, low[1]]).reshape(-1, 32, len(low[0]))      # 32 aux rows a flush
    s = np.zeros((p.shape[0], len(low[0])), dtype=np.float32)
    for r in range(32):
        for _ in range(nocc):
            s = (s + p[:, r]).astype(np.float32)                  # a fused multiply-add rounds once
    want = np.sqrt(np.mean((s.sum(axis=0, dtype=np.float64) / exact - 1) ** 2))
    got = np.sqrt(np.mean((vk.cpu().numpy()[low] / exact - 1) ** 2))
    print(f'  rms relative error {got:.2e}, of FP32 sums of {32 * nocc} products {want:.2e}')
    assert got < 1.2 * want
