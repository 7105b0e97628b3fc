"""The library's host code on the CPU: its sources compiled for the host only and
linked to a stand-in for the HIP runtime (tests/host/hip_stub.cpp) that logs each
launch, event and wait with its stream.  Shown here is what no GPU run shows
reliably: which kernels a call takes, how calls on several streams are ordered
over a shared workspace, and what a call does when memory runs out or a stream is
gone."""
import ctypes
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

import build as pkg_build
import g4hip
import test_gpu_parity as gpu

HERE = os.path.dirname(os.path.abspath(__file__))
Q8_0, Q4_0, Q4_K, Q5_K, Q6_K, F16, BF16 = 8, 2, 12, 13, 14, 1, 30
KERNELS = ["k_split", "k_mm", "k_tok_q4k", "k_tok_reduce", "k_mat", "k_rows", "k_wide", "k_grp_q4k"]


def _run(cmd):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert p.returncode == 0, p.stdout
    return p.stdout


@pytest.fixture(scope="module")
def hip(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("host"))
    host = [pkg_build.HIPCC, "-O1", "-std=c++17", "-fPIC", "-w", "-c"]
    jobs = [host + [os.path.join(HERE, "host", "hip_stub.cpp"), "-o", os.path.join(d, "stub.o")]]
    for src in pkg_build.SOURCES:
        jobs.append(host + ["--offload-host-only", "--offload-arch=" + pkg_build.ARCH, "-I",
                            os.path.join(pkg_build.ROOT, "include"), os.path.join(pkg_build.CSRC, src), "-o",
                            os.path.join(d, src + ".o")])
    with ThreadPoolExecutor(len(jobs)) as ex:
        list(ex.map(_run, jobs))
    objs = [j[-1] for j in jobs]
    # the device code that the host objects refer to is not there
    fat = {w for l in _run(["nm", "-u"] + objs).splitlines() for w in l.split() if w.startswith("__hip_fatbin")}
    so = os.path.join(d, "libg4host.so")
    _run(["g++", "-shared", "-Wl,-Bsymbolic"] + ["-Wl,--defsym=%s=0" % f for f in sorted(fat)] + ["-o", so] + objs)
    L = ctypes.CDLL(so)
    for name, args in g4hip.SIGNATURES.items():
        getattr(L, name).argtypes = args
    L.g4_last_error.restype = L.stub_log.restype = ctypes.c_char_p
    L.stub_free_bytes.argtypes = [ctypes.c_size_t]
    L.stub_capture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    L.stub_stream_id.argtypes = L.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    yield L
    L.stub_free_bytes(ctypes.c_size_t(-1).value)


class Program:
    """One context and a weight of every size asked for; its calls as a program makes them."""

    def __init__(self, hip):
        self.hip, self.weights = hip, {}
        hip.stub_free_bytes(ctypes.c_size_t(-1).value)
        hip.hipGetLastError()
        self.ctx = ctypes.c_void_p()
        assert hip.g4_open(0, ctypes.byref(self.ctx)) == 0
        hip.stub_clear()

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.hip.stub_free_bytes(ctypes.c_size_t(-1).value)
        for w in self.weights.values():
            self.hip.g4_weight_free(w)
        assert self.hip.g4_close(self.ctx) == 0

    def stream(self):
        s = ctypes.c_void_p()
        assert self.hip.hipStreamCreateWithFlags(ctypes.byref(s), 0) == 0
        return s

    def use(self, stream):
        assert self.hip.g4_ctx_set_stream(self.ctx, stream) == 0

    def weight(self, t, elems):
        if (t, elems) not in self.weights:
            n, w = (ctypes.c_int64 * 1)(), (ctypes.c_void_p * 1)()
            assert self.hip.g4_byte_size(t, elems, n) == 0
            assert self.hip.g4_upload(self.ctx, t, ctypes.create_string_buffer(n[0]), n[0], elems, w) == 0
            self.weights[t, elems] = w[0]
        return self.weights[t, elems]

    def batch(self, t, m, rows, cols):
        """matmul_batch_dev; the names of the kernels it launched."""
        w = self.weight(t, rows * cols)
        before = len(self.log())
        rc = self.hip.g4_matmul_batch_dev(self.ctx, w, 0, 4096, m, 8192, rows, cols)
        assert rc == 0, self.hip.g4_last_error()
        return [self.kernel(l[1]) for l in self.log()[before:] if l[0] == "launch"]

    def moe(self, experts, dim, ff, k, tokens):
        """moe_dev; the names of the kernels it launched."""
        gu, dn = self.weight(Q4_K, experts * 2 * ff * dim), self.weight(Q4_K, experts * dim * ff)
        before = len(self.log())
        rc = self.hip.g4_moe_dev(self.ctx, gu, dn, 4096, tokens, dim, ff, 8192, 12288, k, 16384)
        assert rc == 0, self.hip.g4_last_error()
        return [self.kernel(l[1]) for l in self.log()[before:] if l[0] == "launch"]

    def log(self):
        return [l.split() for l in self.hip.stub_log().decode().splitlines()]

    @staticmethod
    def kernel(name):
        return next((k for k in KERNELS if "%d%s" % (len(k), k) in name), name)

    def assert_ordered(self):
        """Every launch that uses a workspace comes after the previous one that used
        the same memory, in stream order or over events and waits of the host."""
        streams, events, host, used, planes = {}, {}, {}, {}, {}

        def merge(a, b):
            for k, v in b.items():
                a[k] = max(a.get(k, 0), v)

        for l in self.log():
            if l[0] == "launch":
                k, s = self.kernel(l[1]), l[2]
                c = streams.setdefault(s, {})
                merge(c, host)
                ws = [l[3]] if len(l) > 3 else []
                if k == "k_split":
                    planes[s] = l[3]
                elif k in ("k_mm", "k_tok_reduce") and s in planes:
                    ws.append(planes[s])  # of its k_split
                for w in ws:
                    for other, n in used.get(w, {}).items():
                        assert c.get(other, 0) >= n, "unordered use of the workspace: %s" % l
                c[s] = c.get(s, 0) + 1
                for w in ws:
                    used[w] = {s: c[s]}
            elif l[0] == "record":
                events[l[1]] = dict(streams.setdefault(l[2], {}))
            elif l[0] == "wait":
                merge(streams.setdefault(l[1], {}), events.get(l[2], {}))
            elif l[0] == "sync":
                merge(host, streams.get(l[1], {}))
            elif l[0] == "sync_event":
                merge(host, events.get(l[1], {}))
            elif l[0] in ("sync_device", "free"):  # (hipFree waits for the device)
                for c in streams.values():
                    merge(host, c)
                if l[0] == "free":
                    used.pop(l[1], None)


# many-token calls that take the tiled product (its planes and split sums are in a
# workspace of the context)
MANY = [(Q6_K, 512, 8192, 2048), (Q4_0, 201, 2048, 8192), (Q4_K, 512, 8192, 2048)]


@pytest.mark.parametrize("t,m,rows,cols", MANY)
def test_many_token_calls_on_several_streams_are_ordered(hip, t, m, rows, cols):
    with Program(hip) as p:
        streams = [None, p.stream(), p.stream()]
        for k in (0, 0, 1, 2, 2, 1, 0, 1):
            p.use(streams[k])
            assert "k_mm" in p.batch(t, m, rows, cols)
        p.assert_ordered()


@pytest.mark.parametrize("same_handle", [False, True])
def test_many_token_calls_after_their_stream_is_gone(hip, same_handle):
    """The stream of the last call has been destroyed: the next call runs all its
    kernels and succeeds, also where the runtime gives the same handle out again
    while that call's work may not be done."""
    with Program(hip) as p:
        a = p.stream()
        b = None if same_handle else p.stream()
        p.use(a)
        p.batch(*MANY[0])
        hip.hipStreamDestroy(a)
        b = b or p.stream()
        assert (a.value == b.value) == same_handle
        p.use(b)
        assert p.batch(*MANY[0]) == ["k_split", "k_mm"]
        p.use(None)
        assert p.batch(*MANY[0]) == ["k_split", "k_mm"]
        assert hip.stub_last_error() == 0
        p.assert_ordered()


def test_many_token_call_without_memory_for_its_workspace(hip):
    with Program(hip) as p:
        p.batch(Q6_K, 2, 8192, 2048)  # (uploads)
        p.hip.stub_free_bytes(1 << 20)
        assert p.batch(Q6_K, 512, 8192, 2048) == ["k_mat"]
        assert p.hip.stub_last_error() == 0


def test_many_token_call_beside_another_streams_capture(hip):
    """A capture on another stream, the one of the last call among them, does not
    change which kernels a call runs."""
    with Program(hip) as p:
        a = p.stream()
        p.use(a)
        p.batch(Q6_K, 2, 16384, 2048)  # (uploads)
        p.batch(*MANY[0])
        p.hip.stub_capture(a, 1)
        p.use(None)
        assert p.batch(*MANY[0]) == ["k_split", "k_mm"]
        assert p.batch(Q6_K, 1024, 16384, 2048) == ["k_split", "k_mm"]
        p.hip.stub_capture(a, 0)
        p.use(a)
        p.batch(*MANY[0])
        p.assert_ordered()


@pytest.mark.parametrize("t,m,rows,cols", [(Q4_K, 512, 2048, 8192), (Q4_K, 512, 4096, 4096), (Q4_K, 201, 2560, 10240),
                                           (Q8_0, 512, 2048, 8192), (Q4_0, 201, 2048, 8192), (Q6_K, 300, 2048, 8192)])
def test_an_eager_call_leaves_the_scratch_for_its_capture(hip, t, m, rows, cols):
    """include/g4hip.h: run the largest shapes once eagerly before capturing.  The
    eager calls here take the tiled product, the captured ones the 16-token tiles
    with their split sums in the scratch."""
    with Program(hip) as p:
        s = p.stream()
        p.use(s)
        assert "k_mm" in p.batch(t, m, rows, cols)
        hip.stub_clear()
        hip.stub_capture(s, 1)
        assert p.batch(t, m, rows, cols) == ["k_tok_q4k" if t == Q4_K else "k_mat", "k_tok_reduce"]
        assert not [l for l in p.log() if l[0] == "malloc"]
        hip.stub_capture(s, 0)


# several tokens on rows of more than 2048 columns: 16-token tiles with column splits
WIDE = [(Q8_0, 12, 2048, 8192), (Q5_K, 40, 4096, 4096), (BF16, 4096, 8192, 8192), (F16, 5, 2048, 8192)]


@pytest.mark.parametrize("t,m,rows,cols", WIDE)
def test_wide_calls_on_several_streams_are_ordered(hip, t, m, rows, cols):
    """Their split sums are in no memory that another stream's call, or a graph, may
    be using."""
    with Program(hip) as p:
        streams = [None, p.stream(), p.stream()]
        for k in (0, 1, 2, 2, 0, 1):
            p.use(streams[k])
            assert p.batch(t, m, rows, cols)[:2] == ["k_mat", "k_tok_reduce"]
        p.assert_ordered()
        used = {l[3] for l in p.log() if l[0] == "launch"}
        # (captured: in the scratch)
        p.use(streams[1])
        hip.stub_capture(streams[1], 1)
        hip.stub_clear()
        assert p.batch(t, m, rows, cols)[:2] == ["k_mat", "k_tok_reduce"]
        assert not used & {l[3] for l in p.log() if l[0] == "launch"}
        hip.stub_capture(streams[1], 0)


@pytest.mark.parametrize("t,m,rows,cols", WIDE)
def test_wide_call_without_memory_for_its_split_sums(hip, t, m, rows, cols):
    with Program(hip) as p:
        p.batch(t, 2, rows, cols)  # (uploads)
        hip.stub_free_bytes(100 << 10)
        assert p.batch(t, m, rows, cols)[0] in ("k_rows", "k_wide")
        assert hip.stub_last_error() == 0
        s = p.stream()
        p.use(s)
        hip.stub_capture(s, 1)
        assert p.batch(t, m, rows, cols)[0] in ("k_rows", "k_wide")
        hip.stub_capture(s, 0)


@pytest.mark.parametrize("t", [Q5_K, BF16, Q8_0])
def test_split_sums_are_bounded(hip, t):
    """4096 tokens x 8192 x 8192: the sums of four splits at once would be 512 MB, in
    the workspace and again in the scratch."""
    with Program(hip) as p:
        p.batch(t, 2, 8192, 8192)
        hip.stub_clear()
        assert p.batch(t, 4096, 8192, 8192).count("k_tok_reduce") >= 8
        assert sum(int(l[1]) for l in p.log() if l[0] == "malloc") <= 2 * (130 << 20)


MAT_TYPES = [Q8_0, Q4_0, Q5_K, Q6_K, BF16, F16]


def test_shapes_meant_for_the_16_token_tiles_take_them(hip):
    """The sizes at which tests/test_gpu_parity.py and its neighbours test k_mat."""
    with Program(hip) as p:
        cases = [(t,) + s[:3] for t in MAT_TYPES for s in gpu.MAT_SHAPES]
        cases += [(t,) + s[:3] for t in (Q8_0, Q4_0) for s in gpu.MAT_ODD_BLOCKS] + gpu.MAT_FEW
        cases += [(t, 12, 2056, 2048) for t in MAT_TYPES]
        cases += [(BF16, 5, 840, 512), (F16, 5, 840, 512), (BF16, 700, 8192, 4160), (Q8_0, 12, 1401, 4096)]
        cases += [(t, m, 2048, 8192) for t in (Q8_0, BF16) for m in (9, 12, 64)]
        cases += [(t, 20, 1248, 2048) for t in (Q4_0, Q5_K)]
        cases += [(Q8_0, 16, 544, 16384), (Q8_0, 16, 528, 32768), (F16, 16, 256, 16384), (BF16, 16, 256, 16384),
                  (BF16, 16, 512, 8192)]
        for c in cases:
            assert p.batch(*c)[0] == "k_mat", c


# (type, tokens, rows, columns), just below and above the outputs from which the
# 16-token tiles are the faster route; the measured times stand at mat_min_tokens
@pytest.mark.parametrize("t,m,rows,cols", [(Q8_0, 8, 1024, 512), (Q8_0, 32, 512, 4096), (Q8_0, 16, 1024, 2048),
                                           (Q8_0, 4, 4096, 2048), (Q8_0, 8, 1024, 8192), (Q4_0, 12, 2048, 2048),
                                           (Q4_0, 6, 4096, 4096), (Q5_K, 16, 1024, 2048), (Q6_K, 16, 1024, 2048),
                                           (Q6_K, 9, 512, 8192), (BF16, 4, 1024, 2048), (F16, 4, 1024, 2048),
                                           (BF16, 4, 512, 8192), (BF16, 9, 512, 3072)])
def test_few_outputs_stay_on_the_row_engine(hip, t, m, rows, cols):
    with Program(hip) as p:
        assert p.batch(t, m, rows, cols)[0] in ("k_rows", "k_wide")
        assert p.batch(t, m + 1 + (t == Q4_0), rows, cols)[0] == "k_mat"


@pytest.mark.parametrize("m,rows,cols", [(256, 4096, 512), (128, 8192, 512), (200, 8192, 1024), (200, 5000, 512),
                                         (400, 4096, 1024)])
def test_short_q4_k_rows_stay_on_the_16_token_tiles(hip, m, rows, cols):
    """Where the tiled product takes 22 to 39% longer."""
    with Program(hip) as p:
        assert p.batch(Q4_K, m, rows, cols) == ["k_tok_q4k"]
        assert "k_mm" in p.batch(Q4_K, 4 * m, rows, cols)


# (experts, columns, ff, slots, tokens)
@pytest.mark.parametrize("shape,grouped", [((128, 1024, 704, 4, 41), False), ((128, 1024, 704, 8, 256), True),
                                           ((32, 2048, 704, 8, 41), True), ((32, 2048, 704, 1, 256), True),
                                           ((128, 2048, 704, 2, 64), False), ((300, 512, 320, 8, 41), False),
                                           ((32, 1024, 320, 1, 256), False), ((32, 1024, 768, 1, 41), True),
                                           ((32, 1024, 768, 8, 40), False)])
def test_grouped_experts_where_they_are_faster(hip, shape, grouped):
    """Both sides' measured times stand at moe_grp_faster."""
    with Program(hip) as p:
        assert ("k_grp_q4k" in p.moe(*shape)) == grouped


def test_shapes_meant_for_the_grouped_experts_take_them(hip):
    with Program(hip) as p:
        for E, D, FF, K, T, *_ in gpu.MOE_STRETCHES:
            assert p.moe(E, D, FF, K, T).count("k_grp_q4k") == 2, (E, D, FF)


def test_a_reservation_covers_the_workspace(hip):
    """A program that reserved up front meets no allocation and no wait of the host in
    its first prompt."""
    with Program(hip) as p:
        for t, m, rows, cols in MANY + WIDE[:2]:
            p.weight(t, rows * cols)
        assert hip.g4_ctx_reserve(p.ctx, 256 << 20) == 0
        hip.stub_clear()
        s = p.stream()
        for k, c in enumerate(MANY + WIDE[:2] + MANY):
            p.use((None, s)[k % 2])
            assert p.batch(*c)[0] in ("k_split", "k_mat")
        assert not [l for l in p.log() if l[0] in ("malloc", "free", "sync", "sync_event", "sync_device")]
        p.assert_ordered()


def test_a_reservation_without_memory_for_the_workspace(hip):
    with Program(hip) as p:
        hip.stub_free_bytes(40 << 20)
        assert hip.g4_ctx_reserve(p.ctx, 32 << 20) == 0
        assert hip.stub_last_error() == 0


def test_shapes_meant_for_the_tiled_product_take_it(hip):
    """The sizes at which tests/test_gpu_parity.py and its neighbours test k_mm."""
    with Program(hip) as p:
        cases = [c[:4] for c in gpu.MM_SHAPES]
        cases += [(t, 512, 8192, 1024) for t in (Q8_0, Q4_0, Q4_K, Q6_K, F16)]
        cases += [(t, 512, 8192, 512) for t in (Q4_0, Q4_K)]
        cases += [(Q6_K, m, 8192, 2048) for m in (100, 300, 120, 1300, 200, 700)]
        cases += [(Q8_0, 512, 512, 32768), (Q4_0, 300, 2048, 8192), (Q6_K, 512, 8192, 2048)]
        for c in cases:
            assert "k_mm" in p.batch(*c), c
        assert p.batch(Q8_0, 1024, 4100, 8192).count("k_mm") == 3  # rows in passes
        assert p.batch(Q6_K, 1300, 8192, 2048).count("k_split") == 2  # tokens in passes
        assert p.batch(Q4_K, 512, 8100, 2048) == ["k_split", "k_mm"]  # no split
