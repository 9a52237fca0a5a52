"""The chunk sweeps of RI-J on the CPU, integrals replaced by the chunk's
name: what the buffer holds when a chunk is contracted."""
import types

import pytest


@pytest.fixture
def sweep(monkeypatch):
    """(state of n chunks, a sweep recording what it contracted, evaluations)"""
    from electrolites_amd import fastdfj3c, ints
    evals = []

    def chunk(ao, aux, tk, blk, width, col_map):
        evals.append(tk.name)
        blk[0] = tk.name
    monkeypatch.setattr(ints, 'int3c2e_chunk', chunk)

    class Buf(list):
        def __getitem__(self, i):
            return self if isinstance(i, slice) else list.__getitem__(self, i)

    def state(n):
        return types.SimpleNamespace(ao=None, aux=None, naux=1, buf=Buf([None]), held=None, tasks=[
            types.SimpleNamespace(name=i, c0=i, c1=i + 1, cmap=None) for i in range(n)])

    def run(st, held=None):
        seen = []
        return fastdfj3c._sweep(st, lambda tk, blk, width: seen.append((tk.name, blk[0])), held), seen
    return state, run, evals


@pytest.mark.parametrize('n', [1, 2, 3])
def test_second_sweep_starts_on_the_held_chunk(sweep, n):
    state, run, evals = sweep
    st = state(n)
    held, seen = run(st)
    assert seen == [(i, i) for i in range(n)]
    _, seen = run(st, held)
    assert seen[0] == (n - 1, n - 1) and sorted(seen) == [(i, i) for i in range(n)]
    assert len(evals) == 2 * n - 1


@pytest.mark.parametrize('n', [1, 2, 3])
@pytest.mark.parametrize('other', ['first', 'both'])
def test_another_call_between_the_sweeps(sweep, n, other):
    """A second thread's call on the same molecule leaves another chunk in
    the shared buffer: the first call contracts its own all the same."""
    state, run, _ = sweep
    st = state(n)
    held, _ = run(st)
    theirs, _ = run(st)
    if other == 'both':
        run(st, theirs)
    _, seen = run(st, held)
    assert sorted(seen) == [(i, i) for i in range(n)]
