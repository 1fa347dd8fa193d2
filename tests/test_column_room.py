"""Which column sweeps may run side by side on one device: all of one call, and
those of several calls as long as two per CU hold them.  Beyond, columns of two
launches could wait for ones that the other launch keeps out of their places."""
import threading

import pytest

from pot3d_amd import _lib

DEV, CUS = 63, 256  # (a device number that no test uses otherwise)


@pytest.fixture
def lib():
    L = _lib.load()
    yield L


def _room(n):
    """Places that n columns take in the worst case, dealt out over 8 XCDs."""
    return -(-n // 8)


def test_one_call_always_finds_room(lib):
    for n in (1, 84, 722, 100000):
        assert lib.p3d_columns_claim(DEV, n, CUS) == 1
        lib.p3d_columns_release(DEV, n)


@pytest.mark.parametrize("first,second", [(84, 84), (722, 1), (1, 722), (289, 289), (256, 256),
                                          (248, 250), (505, 1), (2000, 2000)])
def test_second_call(lib, first, second):
    assert lib.p3d_columns_claim(DEV, first, CUS) == 1
    got = lib.p3d_columns_claim(DEV, second, CUS)
    # never more than two per CU on the fullest XCD; refused well below never
    if _room(first) + _room(second) > 2 * CUS // 8:
        assert got == 0
    if first + second + 14 <= 2 * CUS:
        assert got == 1
    # another device is another room
    assert lib.p3d_columns_claim(DEV - 1, 2000, CUS) == 1
    lib.p3d_columns_release(DEV - 1, 2000)
    if got:
        lib.p3d_columns_release(DEV, second)
    lib.p3d_columns_release(DEV, first)
    assert lib.p3d_columns_claim(DEV, 2000, CUS) == 1  # all given back
    lib.p3d_columns_release(DEV, 2000)


def test_many_threads_never_exceed_the_device(lib):
    lock, held, worst = threading.Lock(), [], [0]

    def work(n):
        for _ in range(2000):
            if lib.p3d_columns_claim(DEV, n, CUS):
                with lock:
                    held.append(n)
                    if len(held) > 1:
                        worst[0] = max(worst[0], sum(_room(h) for h in held))
                with lock:
                    held.remove(n)
                lib.p3d_columns_release(DEV, n)

    ts = [threading.Thread(target=work, args=(n,)) for n in (84, 84, 120, 289, 722, 30)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert worst[0] <= 2 * CUS // 8
    assert lib.p3d_columns_claim(DEV, 2000, CUS) == 1
    lib.p3d_columns_release(DEV, 2000)
