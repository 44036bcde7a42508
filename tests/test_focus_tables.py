"""The matched-filter tables in pieces (focusing.tables): the bits of one piece
over all samples, at piece edges, with rows of no, one and two samples, and the
solver's error from any piece."""
import numpy as np
import pytest

from europaraypaths_amd import focusing


def params(nr, spacing=60.0, aperture=9.0, alt=12000.0):
    dm = focusing.C_PY / 48e6
    return {"rx_window_m": dm * nr, "rx_window_offset_m": alt - 0.3 * dm * nr,
            "rx_sample_rate": 48e6, "aperture": aperture, "spacing": spacing, "altitude": alt,
            "eps_2": 3.15, "frequency": 60e6}


@pytest.mark.parametrize("chunk", [1, 7, 500, 4097])
@pytest.mark.parametrize("nr,spacing,aperture", [(40, 60.0, 9.0), (25, 4000.0, 9.0),
                                                 (9, 60.0, 0.001)])
def test_pieces_give_the_whole(monkeypatch, chunk, nr, spacing, aperture):
    par = params(nr, spacing, aperture)
    monkeypatch.setattr(focusing, "CHUNK", 10 ** 9)
    whole = focusing.tables(par, 0, nr - 1, nr)
    monkeypatch.setattr(focusing, "CHUNK", chunk)
    for a, b in zip(focusing.tables(par, 0, nr - 1, nr), whole):
        assert a.dtype == b.dtype
        np.testing.assert_array_equal(a, b)
    # each row's samples are those of the row alone
    hs, nsx, offs, rows, filt = whole
    for i in (0, nr // 2, nr - 1):
        n, h, rb, mf = focusing.row_tables(par, i, nr)
        assert (n, h) == (nsx[i], hs[i])
        s = slice(offs[i], offs[i] + n)
        np.testing.assert_array_equal(rows[s], np.mod(rb, nr))
        np.testing.assert_array_equal(filt[s], mf.astype(np.complex64))


def test_no_root_in_some_piece(monkeypatch):
    monkeypatch.setattr(focusing, "CHUNK", 16)
    with pytest.raises(ValueError, match="different signs"):
        focusing.tables(params(30, aperture=60.0), 0, 29, 30)
