"""How many workgroups a CSR product is cut into, as the sizes of its workspace tell (one counter each): no GPU needed."""
import pytest

from sparsetir_amd import _lib

UNITS = 256  # compute units


def _workgroups(m, feat, nnz, n=50000):
    """Of one slice of features in one piece."""
    return _lib.lib().stir_csr_spmm_workspace_clear_bytes(m, n, feat, nnz) // 4


@pytest.mark.parametrize("feat,resident,room", [(32, 7, 1024), (47, 7, 1024), (100, 7, 1024), (200, 7, 1024),
                                                (260, 6, 704), (500, 6, 704)])
def test_one_turn_where_it_holds_the_entries(feat, resident, room):
    """A launch that fits one turn of resident workgroups asks for no more of them than there are."""
    m = 60000
    for share in (0.45, 0.7, 0.9, 1.0):
        entries = int(UNITS * resident * room * share)
        if (entries - m) * feat >= 500_000_000:
            continue
        wgs = _workgroups(m, feat, entries - m)
        assert UNITS * 4 < wgs <= UNITS * resident + 3, (feat, entries, wgs)  # sizes are rounded up to four counters


@pytest.mark.parametrize("feat,room", [(32, 1024), (200, 1024), (257, 704), (500, 704)])
def test_no_more_entries_than_there_is_room_for(feat, room):
    """The room in LDS that lets as many workgroups be resident as are asked for; wide rows have less of it."""
    m = 60000
    for entries in range(200_000, min(6_000_000, 500_000_000 // feat + m), 50_000):
        assert entries <= room * _workgroups(m, feat, entries - m), (feat, entries)


@pytest.mark.parametrize("feat,resident,room", [(24, 7, 1024), (47, 7, 1024), (100, 7, 1024), (200, 7, 1024),
                                                (300, 6, 704)])
def test_no_nearly_empty_last_turn(feat, resident, room):
    """A few more entries than one turn of the largest workgroups holds: smaller ones, so that a second turn is worth it."""
    m = 60000
    for share in (1.01, 1.05, 1.1):
        entries = int(UNITS * resident * room * share)
        assert _workgroups(m, feat, entries - m) > 1.3 * UNITS * resident, (feat, share)


@pytest.mark.parametrize("feat,m,nnz", [(256, 169343, 1166243), (192, 150000, 1200000), (512, 40000, 1500000),
                                        (128, 300000, 7800000), (512, 10000, 300000)])
def test_slices_take_several_turns(feat, m, nnz):
    """In slices of 64 features a workgroup takes 768 entries, whatever the turns: neither what it has room for nor a
    share of one turn."""
    slices = feat // 64
    assert abs(_workgroups(m, feat, nnz, n=m) / slices - (m + nnz) / 768) <= 4
