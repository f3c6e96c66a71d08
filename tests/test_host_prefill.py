"""The launches of a prefill call on a model of the device (prefill_model.cpp, compiled for the host with the library's own
kv_api.cpp): every shape that the workspace leaves it, from all layers' tiles kept to one kv head at a time, reads and
writes inside its allocations, finds every key tile written, and attends every row once; a call that the device cannot
hold changes nothing."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qwen38-megakernel_amd", "csrc")
MIB = 1 << 20
P = ctypes.c_void_p
OUT, ANY = 1 << 40, 1 << 41  # addresses of the caller's buffers
F = "K*=5r,V*=6"


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("prefill") / "model.so"
    api = os.environ.get("KV_API_CPP", os.path.join(CSRC, "kv_api.cpp"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__", f'-DKV_API="{api}"', "-I/opt/rocm/include",
                    f"-I{CSRC}", os.path.join(HERE, "prefill_model.cpp"), "-o", str(so)], check=True)
    l = ctypes.CDLL(str(so))
    l.mk_last_error.restype = l.model_faults.restype = ctypes.c_char_p
    l.mk_kv_new.restype = P
    l.mk_kv_new.argtypes = [ctypes.c_char_p] + [ctypes.c_int] * 7
    l.model_used.restype = ctypes.c_size_t
    l.model_room.argtypes = [ctypes.c_size_t, ctypes.c_int]
    l.model_faults.argtypes = [ctypes.c_longlong]
    l.mk_kv_config.argtypes = [P, ctypes.c_char_p, ctypes.c_longlong]
    l.mk_kv_append.argtypes = [P] + [ctypes.c_int] * 5 + [P, P, ctypes.c_int, P]
    l.mk_kv_prefill.argtypes = [P] + [ctypes.c_int] * 5 + [P, P, ctypes.c_int, P, P, P]
    l.model_begin.argtypes = l.mk_free.argtypes = [P]
    l.model_stored.argtypes = [P, ctypes.c_int]
    return l


class Store:
    def __init__(self, lib, spec, win, nl, ctx):
        self.l, self.nl = lib, nl
        lib.model_room(0, 0)
        self.h = lib.mk_kv_new(spec.encode(), win, 0, nl, 1, ctx, 0, 0)
        assert self.h, lib.mk_last_error()

    def append(self, n):
        for p in range(0, n, 4096):
            assert self.l.mk_kv_append(self.h, 0, 0, self.nl, p, min(4096, n - p), ANY, ANY, 0, None) == 0, self.l.mk_last_error()

    def prefill(self, pos, T):
        """-> (appends, launches, most pieces, most layers, fewest kv heads of a launch), or the message of the refusal"""
        self.l.model_begin(OUT)
        if self.l.mk_kv_prefill(self.h, 0, 0, self.nl, pos, T, ANY, ANY, 0, ANY, OUT, None) < 0:
            return self.l.mk_last_error().decode()
        faults = self.l.model_faults(4 * self.nl * T).decode()
        assert faults == "", faults
        c = (ctypes.c_int * 5)()
        self.l.model_counts(c)
        return tuple(c)

    def stored(self):
        return self.l.model_stored(self.h, 0)

    def close(self):
        self.l.model_room(0, 0)
        self.l.mk_free(self.h)


# (spec, window, layers, stored, tokens): one bucket and several, a prompt, groups past a window, the ring of window tiles
# wrapped (182 tiles, 5,824 positions), windows as long as a group or shorter
CALLS = [("", 0, 4, 0, 1111), (F, 2048, 2, 0, 7000), (F, 2048, 2, 6001, 4000), ("K*=6,V*=4r", 512, 3, 5000, 3000), (F, 640, 1, 1279, 2),
         (F, 2048, 1, 60001, 1500), ("K0=5,V*=5,K1=6,K2=6", 1024, 4, 650, 1300)]


@pytest.mark.parametrize("spec,win,nl,pos,T", CALLS)
def test_every_shape_covers_the_call(lib, spec, win, nl, pos, T):
    seen, room = set(), 0
    while 0 not in seen:
        st = Store(lib, spec, win, nl, pos + T)
        st.append(pos)
        assert lib.mk_kv_config(st.h, b"prefill_scratch", room) == 0
        used = lib.model_used()
        r = st.prefill(pos, T)
        if isinstance(r, str):  # the least it can work in is more than the bound
            assert "no device memory" in r and st.stored() == pos and lib.model_used() == used
            seen.add(0)
        else:
            assert st.stored() == pos + T and (not room or lib.model_used() - used <= room)
            seen.add(r[4])
            room = (lib.model_used() - used) * 9 // 10
        st.close()
    assert seen == {4, 2, 1, 0}, seen


def test_full_device(lib):
    # the memory is short for real, not by the knob: what is left is enough for one layer's tiles, not for four pieces' partials
    st = Store(lib, F, 2048, 1, 16384)
    used = lib.model_used()
    lib.model_room(200 * MIB, 0)
    r = st.prefill(0, 16384)
    assert r[0] == 26 and lib.model_used() - used <= 200 * MIB  # (26 buckets: one piece at a time)
    st.close()
    # nothing is left: nothing is stored, launched or kept
    st = Store(lib, F, 2048, 1, 16384)
    used = lib.model_used()
    lib.model_room(20 * MIB, 0)
    assert "no device memory" in st.prefill(0, 16384)
    c = (ctypes.c_int * 5)()
    lib.model_counts(c)
    assert st.stored() == 0 and c[0] == c[1] == 0 and lib.model_used() == used
    # and with the memory back, the same call runs
    lib.model_room(0, 0)
    assert st.prefill(0, 16384)[2] == 4
    st.close()


def test_other_errors_are_reported_as_they_are(lib):
    st = Store(lib, F, 2048, 2, 2000)
    lib.model_room(0, 401)  # hipErrorIllegalState: no smaller call would help
    r = st.prefill(0, 2000)
    assert "illegal state" in r and "no device memory" not in r and st.stored() == 0
    st.close()


def test_a_longer_context_inside_a_capture(lib):
    # warmed up on the first chunk; the captured one reads 40 times as many keys
    st = Store(lib, F, 2048, 1, 50000)
    st.prefill(0, 640)
    st.append(40000)
    lib.model_capture(1)
    r = st.prefill(40000, 640)
    assert lib.model_capture(0) == 1  # (the thread's capture mode as it was)
    assert r[4] == 4 and st.stored() == 40640, r
    st.close()


def test_a_short_prompt_with_a_large_window(lib):
    # 16 tokens over 16 layers: two tiles of each kind per layer and head, not the 362 that the window can have
    st = Store(lib, F, 8192, 16, 20000)
    used = lib.model_used()
    r = st.prefill(0, 16)
    assert r[1:4] == (2, 1, 16), r  # all layers' tiles in one launch, all layers in one attention
    # (and three blocks of 32 query rows per head: 64 workgroups)
    assert lib.model_used() - used == 16 * 4 * ((2 + 2) * 32768 + 3 * 16384)
    st.close()


def test_the_tiles_grow_within_their_bound(lib):
    # 586 MiB of tiles, then 601: asked for ahead of the need, but not past 640 MiB (the outgrown buffer is kept beside it)
    st = Store(lib, "", 0, 4, 40000)
    st.append(37500)
    used = lib.model_used()
    st.prefill(37500, 1)
    first = lib.model_used() - used
    assert 586 * MIB < first < 600 * MIB
    st.append(38400)
    st.prefill(38400, 1)
    assert lib.model_used() - used - first <= 641 * MIB
    st.close()


@pytest.mark.parametrize("pos,T,groups,own", [(500, 16, 1, 0), (1072, 128, 1, 0), (3199, 1, 1, 0), (6001, 399, 1, 0), (6400, 640, 1, 0),
                                              (600, 2600, 2, 0), (6001, 400, 1, 0), (6001, 440, 1, 1), (6001, 1000, 1, 1), (2000, 4000, 2, 1)])
def test_window_rows_with_the_first_group(lib, pos, T, groups, own):
    # the window's rows before the call take a launch of their own only where the first group's rows replace some of them in
    # the ring of 3,232 (6,001 positions: the window starts at 3,200); otherwise a group is one launch over the tiles and one of
    # the attention.  (That no row is read after it was replaced: as in test_every_shape_covers_the_call.)
    st = Store(lib, F, 2048, 1, pos + T)
    st.append(pos)
    r = st.prefill(pos, T)
    assert r[:2] == (groups, 2 * groups + own), r
    st.close()


@pytest.mark.parametrize("spec,win,nl,pos,T", [(F, 2048, 1, 0, 2000), (F, 2048, 2, 0, 9000), (F, 2048, 1, 30000, 100), (F, 2048, 1, 6001, 4000),
                                               (F, 640, 1, 650, 1300), ("", 0, 4, 1000, 3000), (F, 2048, 16, 12000, 700)])
def test_every_unpacked_tile_is_read(lib, spec, win, nl, pos, T):
    # a window's rows are read from its own tiles: no main tiles are unpacked for them.  (One tile of window rows per layer and
    # head is unpacked twice where those before the call come first: the one that the call's first rows complete.)
    st = Store(lib, spec, win, nl, pos + T)
    st.append(pos)
    assert isinstance(st.prefill(pos, T), tuple)
    assert lib.model_unread() <= 4 * nl * (win > 0 and pos % 32 != 0)
    st.close()


def test_a_short_prompt_takes_one_buffer(lib):
    # rows of one key segment have no partials: their prepared queries take room behind the tiles, not a buffer of their own
    st = Store(lib, F, 2048, 2, 1280)
    n = lib.model_allocations()
    assert isinstance(st.prefill(0, 100), tuple)
    assert lib.model_allocations() - n == 1
    st.close()
