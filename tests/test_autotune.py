"""CPU tests of which tuned entry a solver takes: the shipped table's on the grid it was tuned on, a user's own for its
class of sizes, and the library's choice, which every tuning compares with, otherwise."""
import pytest

from pfkit import _lib, autotune


def _args(nx, ny, nz, k=20):
    return dict(Nx=nx, Ny=ny, Nz=nz, num_oris=k)


@pytest.fixture
def no_user_cache(monkeypatch):
    autotune._load()
    monkeypatch.setattr(autotune, "_cache", {})


@pytest.mark.parametrize("dtype,want", [(_lib.PF_F32, (4, 0x10010)), (_lib.PF_BF16, (3, 0x10010)), (_lib.PF_F64, (2, 0x10016))])
def test_shipped_entries_hold_for_their_grid_alone(no_user_cache, dtype, want):
    assert autotune.lookup(dtype, _args(256, 256, 64), True) == want
    for dims in ((203, 197, 59), (150, 140, 50), (129, 129, 33), (256, 255, 64), (64, 256, 256)):
        assert autotune.lookup(dtype, _args(*dims), True) == (-1, 0)


def test_batches_keep_their_entries(no_user_cache):
    assert autotune.lookup(_lib.PF_F32, _args(40, 33, 20), True, throughput=True) == (2, 6)
    assert autotune.lookup(_lib.PF_F64, _args(40, 33, 20), True, throughput=True) == (2, 0x10016)
    assert autotune.lookup(_lib.PF_F64, _args(40, 33, 20, 16), True, throughput=True) == (-1, 0)


def test_a_users_entry_holds_for_its_class_and_goes_first(no_user_cache):
    autotune._cache[autotune.key(_lib.PF_F32, 20, True, 59, 197, 203)] = dict(tile=1, zchunk=7, ms=0.1)
    for dims in ((203, 197, 59), (256, 256, 64), (130, 140, 40)):
        assert autotune.lookup(_lib.PF_F32, _args(*dims), True) == (1, 7)
    autotune._cache[autotune.key(_lib.PF_F32, 20, True, 59, 197, 203)] = dict(tile=-1, zchunk=0, ms=0.1)
    assert autotune.lookup(_lib.PF_F32, _args(256, 256, 64), True) == (-1, 0)


def test_tuning_compares_with_the_librarys_choice(tmp_path, monkeypatch):
    for dtype, k, nz in ((_lib.PF_F32, 20, 64), (_lib.PF_F64, 33, 1), (_lib.PF_BF16, 7, 5)):
        assert (-1, 0) in autotune.candidates(dtype, k, nz)
    entries = {"a": dict(tile=1, zchunk=2), "b": dict(tile=1, zchunk=2)}
    autotune._put(entries, "a", dict(tile=-1, zchunk=0))
    autotune._put(entries, "b", dict(tile=3, zchunk=4))
    assert entries == {"b": dict(tile=3, zchunk=4)}
