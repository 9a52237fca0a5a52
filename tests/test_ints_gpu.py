"""GPU parity of the generated Rys integral kernels against the
McMurchie-Davidson oracle (an independent algorithm)."""
import numpy as np
import pytest

from oracle import oracle as O


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.fixture(scope='module')
def mol():
    from electrolites_amd.gto import water_cluster
    # two waters and a Li+: every orbital class (s, p, d) and aux l = 0..4
    return water_cluster(2, seed=3, side=5.0, li=True)


@pytest.mark.gpu
def test_int2c2e(mol):
    from electrolites_amd import ints
    aux = ints.DeviceBasis(mol.aux)
    got = ints.int2c2e(aux).cpu().numpy()
    ref = O.int2c2e(mol.aux.as_dict())
    assert rel(got, ref) < 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize('nchunk', [1, 3])
def test_int3c2e(mol, nchunk):
    import torch
    from electrolites_amd import ints
    ao = ints.DeviceBasis(mol.ao)
    aux = ints.DeviceBasis(mol.aux)
    nao, naux = mol.nao, mol.naux
    npairs = nao * (nao + 1) // 2
    full = torch.zeros((naux, npairs), dtype=torch.float64, device='cuda')
    bounds = np.linspace(0, mol.ao.nbas, nchunk + 1).astype(int)
    for I0, I1 in zip(bounds[:-1], bounds[1:]):
        t = ints.PairTasks(mol.ao, I0, I1)
        blk = torch.zeros((naux, t.p1 - t.p0), dtype=torch.float64, device='cuda')
        ints.int3c2e_chunk(ao, aux, t, blk, blk.stride(0))
        full[:, t.p0:t.p1] = blk
    got = full.cpu().numpy()
    j3c = O.int3c2e(mol.ao.as_dict(), mol.aux.as_dict())
    rows, cols = np.tril_indices(nao)
    ref = j3c[rows, cols, :].T
    assert rel(got, ref) < 1e-13


def _metric_and_chunk(mol):
    """A call that evaluates both integral tensors into buffers of its own on
    the current stream, and those buffers."""
    import torch
    from electrolites_amd import ints
    ao, aux = ints.DeviceBasis(mol.ao), ints.DeviceBasis(mol.aux)
    t = ints.PairTasks(mol.ao, 0, mol.ao.nbas)
    t.dev

    def buffers():
        return (torch.zeros((mol.naux, mol.naux), dtype=torch.float64, device='cuda'),
                torch.zeros((mol.naux, t.p1 - t.p0), dtype=torch.float64, device='cuda'))

    def run(out):
        ints.int2c2e(aux, out[0])
        ints.int3c2e_chunk(ao, aux, t, out[1], out[1].stride(0))
        return out
    return buffers, run


@pytest.mark.gpu
def test_callers_on_streams_of_their_own(mol):
    """The integral classes spread over side streams of the caller's: more
    callers' streams than there are sets of them, two threads at a time, each
    behind work on its own stream and read by it afterwards, give the null
    stream's values."""
    import threading
    import torch
    buffers, run = _metric_and_chunk(mol)
    ref = run(buffers())
    torch.cuda.synchronize()
    bad = []

    def caller(streams):
        x = torch.randn(1024, 1024, dtype=torch.float64, device='cuda')
        for s in streams:
            with torch.cuda.stream(s):
                for _ in range(2):
                    out = buffers()
                    for b in out:
                        b.fill_(float('nan'))
                    x @ x
                    for b in out:
                        b.zero_()
                    run(out)
                    if not all(bool(torch.equal(a, b)) for a, b in zip(out, ref)):
                        bad.append(s)
    threads = [threading.Thread(target=caller, args=([torch.cuda.Stream() for _ in range(7)],)) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.gpu
def test_capturing_caller(mol):
    """A captured call stays on its stream: every replay, with eager calls on
    the same buffers between, gives the eager values."""
    import torch
    buffers, run = _metric_and_chunk(mol)
    ref = run(buffers())
    out = run(buffers())
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run(out)
    for rep in range(3):
        for b in out:
            b.fill_(float('nan'))
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, ref)), rep
        run(out)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, ref)), rep


@pytest.mark.gpu
def test_metric_prefactor_precision():
    """The metric's (s|s) entries of one centre are the prefactor alone, 2
    pi^(5/2) / (p q sqrt(p + q)) c_p c_q / 4 pi: over random exponents their
    root mean square error against 80-bit values is that of this expression in
    64 bits with a single division (a product of reciprocals rounds three more
    times, 1.14 times the error)."""
    from electrolites_amd import ints
    from electrolites_amd.gto import water_cluster
    mol = water_cluster(24, seed=3, li=True)
    mol.aux.exps[:] *= np.random.default_rng(0).uniform(.7, 1.3, len(mol.aux.exps))
    aux = mol.aux.as_dict()
    got = ints.int2c2e(ints.DeviceBasis(mol.aux)).cpu().numpy()
    ld = np.longdouble
    pi = ld('3.14159265358979323846264338327950288')
    s = np.flatnonzero((aux['l'] == 0) & (aux['nprim'] == 1))
    i, j = (x[aux['atom'][s][:, None] == aux['atom'][s]] for x in np.broadcast_arrays(s[:, None], s[None]))
    (p, cp), (q, cq) = ((aux['exps'][k], aux['coefs'][k]) for k in (aux['prim_off'][i], aux['prim_off'][j]))
    exact = 2 * pi ** ld(2.5) / (ld(p) * ld(q) * np.sqrt(ld(p) + ld(q))) * ld(cp) * ld(cq) / (4 * pi)
    f64 = 34.986836655249725 / (p * q * np.sqrt(p + q)) * cp * cq * .28209479177387814 * .28209479177387814
    err, sim = (float(np.sqrt(np.mean((x / exact - 1) ** 2))) for x in (got[aux['ao_off'][i], aux['ao_off'][j]], f64))
    print(f'(s|s) prefactor over {len(i)} pairs: rms {err:.3e}, of the 64-bit expression {sim:.3e}', flush=True)
    # the rms of n errors is within n^-1/2 of its mean
    assert len(i) > 3000 and err < 1.04 * sim
