"""First calls of the memory, copy, stream and event entry points from several
threads: the function object a thread calls has its argument types set once,
before any thread can get hold of it (stub library, no device)."""
import threading

from simwave_amd import hipmem


class StubFunction:
    """Stands for a ctypes function: counts the settings of its argument types,
    each of which waits for the other threads to reach theirs."""

    def __init__(self, lib):
        self.lib, self.sets, self.restype = lib, 0, None

    @property
    def argtypes(self):
        return None

    @argtypes.setter
    def argtypes(self, types):
        self.sets += 1
        self.lib.setting.set()
        self.lib.second.wait(0.5)

    def __call__(self, *args):
        self.lib.called.append((self, self.sets, self.restype))
        return 0


class StubLibrary:
    """Stands for a ctypes.CDLL: lib[name] makes a function object, lib.name
    makes it once and keeps it."""

    def __init__(self):
        self.setting, self.second, self.called = threading.Event(), threading.Event(), []

    def __getitem__(self, name):
        return StubFunction(self)

    def __getattr__(self, name):
        if not name.startswith("simwave_hip"):
            raise AttributeError(name)
        fn = self[name]
        setattr(self, name, fn)
        return fn


def test_first_calls_from_two_threads_set_types_once():
    lib = StubLibrary()

    def first():
        hipmem._call(lib, "simwave_hip_stream_synchronize", None)

    def late():
        lib.setting.wait(10)
        threading.Timer(0.1, lib.second.set).start()
        hipmem._call(lib, "simwave_hip_stream_synchronize", None)
    threads = [threading.Thread(target=f) for f in (first, late)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(10)
    assert len(lib.called) == 2
    for fn, sets, restype in lib.called:
        assert sets == fn.sets == 1 and restype is not None


def test_each_library_has_functions_of_its_own():
    a, b = StubLibrary(), StubLibrary()
    for lib in (a, b, a):
        lib.second.set()
        hipmem._call(lib, "simwave_hip_zero", None, 0, None)
    assert len(a.called) == 2 and a.called[0][0] is a.called[1][0]
    assert len(b.called) == 1 and b.called[0][0] is not a.called[0][0]
