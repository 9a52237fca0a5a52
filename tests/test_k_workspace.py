"""The workspace of the exchange on the CPU (the query needs no device)."""
import pytest


@pytest.mark.parametrize('query', ['mdf_get_k_workspace', 'mdf_get_k_tiles_workspace'])
@pytest.mark.parametrize('prec,elem', [(0, 8), (1, 4), (2, 4)])
@pytest.mark.parametrize('two', [0, 1])
@pytest.mark.parametrize('naux', [5, 37])
def test_passes_keep_the_bound(monkeypatch, query, prec, elem, two, naux):
    """The transformed blocks of a pass take no more than the bound allows
    (MDF_K_BLOCK_BYTES, or a caller's number of rows), down to one row."""
    from electrolites_amd import _lib
    nao, nocc = 16, 100_000
    # beside the blocks: at most 256 partials, packed factors or split planes
    # of rows rounded up to 320 columns, row strides rounded up to 4, 256-byte pieces
    rest = 256 * nao * nao * 8 + (1 + two) * ((nao + 17) * (nocc + 320) * elem + 8 * nao * 4 * elem + 4096)
    row = nao * nocc * elem * (1 + two)
    last = 0
    for rows in range(1, 45):
        monkeypatch.setenv('MDF_K_BLOCK_BYTES', str(rows * row))
        bound = _lib.query(query, naux, nao, nocc, two, prec, 0)
        monkeypatch.delenv('MDF_K_BLOCK_BYTES')
        asked = _lib.query(query, naux, nao, nocc, two, prec, rows)
        assert bound <= rows * row + rest and asked <= rows * row + rest, rows
        last = asked
    assert last >= naux * row, 'every row in one pass once they fit'
