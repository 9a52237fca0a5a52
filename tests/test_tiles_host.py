"""Host side of the pair tiles on the CPU, with the library and the streams
replaced: when tiles are built, when they may be used, what is kept."""
import types

import pytest


class FakeStream:
    cuda_stream = 7

    def __init__(self, log):
        self.log = log

    def synchronize(self):
        self.log.append('sync')


class FakeEvent:
    def __init__(self, *a, **k):
        pass

    def record(self, *a):
        pass

    def query(self):
        return False


@pytest.fixture
def fake(monkeypatch):
    """The library's calls and the stream's waits, in order; ``capturing``
    says whether the current stream is being captured."""
    import torch
    from electrolites_amd import _dev, _lib
    f = types.SimpleNamespace(log=[], capturing=False)
    stream = FakeStream(f.log)
    monkeypatch.setattr(_lib, 'query', lambda name, *a: f.log.append(name) or 4096)
    monkeypatch.setattr(_lib, 'call', lambda name, *a: f.log.append(name))
    monkeypatch.setattr(_dev, 'stream_ptr', lambda: None)
    monkeypatch.setattr(_dev, 'device', lambda: torch.device('cpu'))
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda *a: stream)
    monkeypatch.setattr(torch.cuda, 'is_current_stream_capturing', lambda: f.capturing)
    monkeypatch.setattr(torch.cuda, 'Event', FakeEvent)
    return f


def layout(nao=120):
    """A screened layout: the last pair of the triangle is not stored."""
    import numpy as np
    from electrolites_amd import fastdf
    rows, cols = np.tril_indices(nao)
    addr = (rows * nao + cols).astype(np.int32)[:-1]
    return fastdf._PairLayout(addr, nao, len(addr))


@pytest.mark.parametrize('via', ['entry', 'layout', 'lower'])
def test_tiles_are_complete_when_handed_out(fake, via):
    """Whoever gets the tiles may run on any stream: the host has waited for
    the build by then."""
    import torch
    from electrolites_amd import batch
    lay = layout()
    if via == 'entry':
        buf = batch.Entry(torch.zeros(3, lay.npairs, dtype=torch.float64), 120, 1, 2, pair_map=lay.map).tiles()
    else:
        buf = lay.tiles(lower=via == 'lower')
    assert buf is not None
    assert 'sync' in fake.log[fake.log.index('mdf_build_pair_tiles'):]


def test_a_captured_call_builds_no_tiles(fake):
    """Tiles built inside a capture would hold nothing until the graph runs,
    and lie in its memory: the captured call goes without, and a later call
    builds them; once built, a captured call takes them."""
    lay = layout()
    fake.capturing = True
    n = len(fake.log)
    assert lay.tiles() is None and lay.tiles(lower=True) is None
    assert fake.log[n:] == []
    fake.capturing = False
    buf = lay.tiles()
    assert buf is not None
    fake.capturing = True
    assert lay.tiles() is buf and lay.tiles(lower=True) is None


@pytest.mark.parametrize('built', [False, True])
@pytest.mark.parametrize('how', ['deepcopy', 'pickle'])
def test_a_layout_can_be_copied(fake, how, built):
    """As a DF object that keeps one is: the copy has the pair tables and no
    tiles, and the original keeps its own."""
    import copy
    import pickle
    from electrolites_amd import fastdf
    for lay in (layout(), fastdf._PairLayout(None, 4, 10)):
        tiles = lay.tiles() if built else None
        got = copy.deepcopy(lay) if how == 'deepcopy' else pickle.loads(pickle.dumps(lay))
        assert (got.nao, got.npairs, got.full) == (lay.nao, lay.npairs, lay.full)
        assert (got.map is None) == (lay.map is None) and got._tiles == {}
        if tiles is not None:
            assert lay.tiles() is tiles and got.tiles() is not tiles


def test_sizes_the_tiles_do_not_hold(fake):
    """From 2^29 pairs on no tiles are built."""
    from electrolites_amd import fastdf
    pmap = layout().map
    assert fastdf.PairTiles(pmap, 32768, 1 << 29).buf is None
    assert fastdf.PairTiles(pmap, 111, 6000).buf is None
    assert 'mdf_build_pair_tiles' not in fake.log


@pytest.mark.parametrize('nao,npairs', [(32768, 1 << 29), (32769, 100)])
def test_the_library_refuses_them(nao, npairs):
    """Checked before any device call."""
    from electrolites_amd import _lib
    p = 256                                   # a pointer that is not read
    with pytest.raises(Exception, match='pair tiles hold up to'):
        _lib.call('mdf_get_k_tiles', p, 0, 1, npairs, npairs, p, p, nao, p, None, 1, 1, 0, p, nao, 0, p, 1 << 40, None)
    with pytest.raises(Exception, match='pair tiles hold up to'):
        _lib.call('mdf_k_step1_tiles', p, 0, 1, npairs, npairs, p, 0, nao, p, 1, 1, p, 1, nao, p, 1 << 40, None)
