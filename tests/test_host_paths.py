"""What the bridge's host code launches, without a GPU: the library over a HIP
runtime of the test's own (hip_stub.cpp) that records launches and allocations.
Each check runs in a process of its own, since a process binds one runtime."""
from __future__ import annotations

import ctypes as C
import re
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve()
CHECKS = {}


def check(fn):
    CHECKS[fn.__name__] = fn
    return fn


@pytest.fixture(scope="session")
def stub(tmp_path_factory):
    so = tmp_path_factory.mktemp("hip_stub") / "libhip_stub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-DNNC_STUB_SYMBOL_BYTES={32 << 20}", str(HERE.parent / "hip_stub.cpp"), "-o", str(so)], check=True)
    return so


class Runtime:
    def __init__(self, so: str):
        self.lib = C.CDLL(so, mode=C.RTLD_GLOBAL)  # before libnnc_hip.so is loaded
        self.lib.stub_name.restype = C.c_char_p
        self.lib.stub_pointer.restype = C.c_void_p
        self.lib.stub_bytes_left.restype = C.c_size_t
        self.lib.stub_bytes_left.argtypes = [C.c_void_p]
        self.lib.stub_live_bytes.restype = C.c_size_t

    def launches(self):
        """(name, gemv fields, captured) of the launches since the last call of clear()."""
        got = []
        for i in range(self.lib.stub_launches()):
            v = (C.c_int * 5)()
            self.lib.stub_gemv(i, v)
            got.append(dict(zip(("n_batch", "cols", "rows", "x_tiles", "n_split"), v), name=self.lib.stub_name(i).decode(),
                            captured=bool(self.lib.stub_captured(i)), xs=self.lib.stub_pointer(i, 0),
                            scratch=[p for p in (self.lib.stub_pointer(i, w) for w in range(4)) if p]))
        return got

    def clear(self):
        self.lib.stub_clear()

    def left(self, p):
        return self.lib.stub_bytes_left(p)

    def capture(self, fn):
        self.lib.stub_capture(1)
        try:
            fn()
        finally:
            self.lib.stub_capture(0)
        assert not self.lib.stub_capture_invalid(), "a call that a capture does not allow"


FORMATS = ("bf16", "q8_0", "q4_s")


def gemv(kv, fmt, n, rows, cols):
    """(addresses are not read: nothing runs)"""
    kv.gemv_device(fmt, (1 << 20, 2 << 20, 3 << 20), 4 << 20, 5 << 20, rows=rows, cols=cols, n_batch=n)


@check
def staged_x_stays_in_its_allocation(rt, nh):
    """Every 16-vector tile that a gemv kernel reads is one that was staged (the
    kernel of up to 64 vectors reads as many as its instance has; the tile
    kernel clamps), and the staged X fits its allocation, for every number of
    vectors up to 64 and some above."""
    for fmt in FORMATS:
        for cols in (32, 512, 2048, 2560):
            for rows in (16, 1000, 5136):
                for n in (*range(2, 66), 80, 129, 1024):
                    with nh.KVCache([16], [64]) as kv:
                        rt.clear()
                        gemv(kv, fmt, n, rows, cols)
                        for l in rt.launches():
                            if not l["xs"]:
                                continue
                            what = (fmt, cols, rows, n, l["name"])
                            assert l["x_tiles"] == (n + 15) // 16, what
                            nb = cols // 32
                            need = l["x_tiles"] * (nb * 2048 + ((nb + 31) // 32 * 3072 if fmt == "q4_s" else 0))
                            assert need <= rt.left(l["xs"]), what
                            m = re.search(r"gemv_batch_kernelILi\d+ELi\d+ELi(\d+)E", l["name"])
                            if m:
                                assert int(m[1]) <= l["x_tiles"], what


def route(launches):
    """(kernel without its sizes, vectors, K splits) of each launch."""
    return [(re.search(r"gemv_(?:[a-z]+_)*kernel", l["name"])[0], l["n_batch"], l["n_split"]) for l in launches]


@check
def many_vectors_of_few_wide_rows(rt, nh):
    """Where a work-group per tile would leave the chip idle the vectors run 64 or
    16 at a time; and a group's matrices go the way of their own calls."""
    with nh.KVCache([16], [64]) as kv:
        def launched(fmt, rows, cols, n):
            rt.clear()
            if isinstance(rows, int):
                gemv(kv, fmt, n, rows, cols)
            else:
                kv.gemv_group_device(fmt, [((1 << 20, 2 << 20, 3 << 20)[:1 + FORMATS.index(fmt)], 5 << 20, r) for r in rows],
                                     4 << 20, cols=cols, n_batch=n)
            return route(l for l in rt.launches() if "stage_x" not in l["name"] and "reduce" not in l["name"])

        for fmt in FORMATS:
            for n in (65, 80, 96, 97, 112, 113):
                got = launched(fmt, 1024, 9728, n)
                if n <= (96 if fmt == "bf16" else 112):
                    assert got[0][:2] == ("gemv_batch_kernel", 64) and sum(g[1] for g in got) == n, (fmt, n, got)
                else:
                    assert got == [("gemv_tile_kernel", n, 1)], (fmt, n, got)
            assert launched(fmt, 8192, 9728, 80) == [("gemv_tile_kernel", 80, 1)]
            assert launched(fmt, 1024, 2560, 80) == [("gemv_tile_kernel", 80, 1)]
        assert [g[:2] for g in launched("bf16", 640, 9728, 32)] == [("gemv_kernel", 16)] * 2
        for fmt in FORMATS:
            for cols in (512, 1024, 2560, 6144, 9728, 16384):
                for n in (2, 8, 9, 16, 17, 40, 64, 65, 100, 130, 1030):
                    for rows in ((4096, 1024, 1024), (1024, 1024), (1040, 3072, 16), (32000, 1024), (16, 32000)):
                        alone = [launched(fmt, r, cols, n) for r in rows]
                        group = launched(fmt, rows, cols, n)
                        want = alone[0] if all(a == alone[0] for a in alone) else [x for a in alone for x in a]
                        assert group == want, (fmt, cols, n, rows, group, alone)


@check
def narrow_batches_are_one_launch(rt, nh):
    """Up to 16 vectors of at most 256 (BF16) or 384 columns: one launch, no
    scratch; beside the lines X is staged."""
    for fmt in FORMATS:
        last = 256 if fmt == "bf16" else 384
        for cols in (32, 64, last, last + 32):
            for n in (2, 3, 16):
                with nh.KVCache([16], [64]) as kv:
                    rt.clear()
                    gemv(kv, fmt, n, 1000, cols)
                    got = rt.launches()
                    if cols <= last:
                        assert route(got) == [("gemv_kernel", n, 1)] and not got[0]["scratch"], (fmt, cols, n)
                    else:
                        assert [r[0] for r in route(got)] == ["gemv_stage_x_kernel", "gemv_batch_kernel"], (fmt, cols, n)


@check
def few_vectors_of_tall_bf16_matrices(rt, nh):
    """Matrices of many rows keep gemv_kernel up to eight vectors from a number of
    columns on, and 20 000 rows for any number where one K split takes them all."""
    with nh.KVCache([16], [64]) as kv:
        for rows, from_cols in ((6143, 2080), (6144, 1664), (8703, 1664), (8704, 1152), (10752, 1152), (10753, 1664),
                                (19999, 1664), (20000, 864), (151936, 864)):
            for cols in (320, 512, 544, 640, 832, 864, 1120, 1152, 1632, 1664, 2048, 2080):
                for n in (2, 8, 9, 16):
                    rt.clear()
                    gemv(kv, "bf16", n, rows, cols)
                    kernel = [r[0] for r in route(rt.launches()) if "stage_x" not in r[0]][0]
                    split = cols > 2048 or rows >= 20000 and cols <= 512 or n <= 8 and cols >= from_cols
                    assert kernel == ("gemv_kernel" if split else "gemv_batch_kernel"), (rows, cols, n, kernel)
            rt.clear()
            gemv(kv, "q8_0", 2, rows, 1664)
            assert route(rt.launches())[-1][0] == "gemv_batch_kernel"


@check
def captured_batch_with_a_rest(rt, nh):
    """A captured batch of whole launches and a rest finds the scratch of both
    there, or runs a vector at a time: here the staged X of 1024 vectors was
    reserved, and the rest of 16 needs more for its K splits."""
    for warm in (1024, 1040):
        with nh.KVCache([16], [64]) as kv:
            gemv(kv, "bf16", warm, 1 << 16, 2560)
            rt.clear()
            rt.capture(lambda: gemv(kv, "bf16", 1040, 1 << 16, 2560))
            got = {r[:2] for r in route(rt.launches())}
            assert (got == {("gemv_vec_kernel", 1)}) == (warm == 1024), (warm, got)


def attend(kv, n_tok, pos0=0, *, n_head=8, n_kv=8, head_dim=64, causal=True, window=0):
    kv.attend_device(0, 1 << 20, 2 << 20, n_tok=n_tok, pos0=pos0, n_head=n_head, n_kv=n_kv, head_dim=head_dim, scale=0.1,
                     causal=causal, window=window)


@check
def long_f32_batches_take_the_kernel_that_is_faster(rt, nh):
    """The three-part products from enough work on, and only where their operands
    leave room for the splits that fill the chip."""
    three = [(32, 8, 64, 0, 512, True, 0), (8, 8, 128, 0, 1024, True, 0), (3, 1, 256, 0, 2048, False, 512),
             (4, 1, 256, 0, 1000, True, 0), (32, 8, 128, 0, 768, True, 0), (8, 2, 256, 0, 2048, False, 0),
             (16, 8, 128, 0, 2048, True, 0), (32, 8, 64, 2000, 2048, True, 0),
             (8, 2, 256, 0, 1500, False, 0)]
    fp32 = [(32, 8, 64, 0, 300, True, 0), (16, 8, 128, 0, 300, True, 0), (8, 8, 128, 0, 512, False, 0),
            (8, 8, 128, 2000, 512, True, 0), (16, 8, 128, 2000, 512, True, 0), (8, 8, 256, 0, 1024, True, 0),
            (8, 2, 256, 2000, 1024, True, 0), (4, 1, 256, 0, 999, True, 0)]
    for cases, kernel in ((three, "tiled3_kernel"), (fp32, "12tiled_kernel")):
        for n_head, n_kv, hd, pos0, n, causal, window in cases:
            with nh.KVCache([4096], [n_kv * hd], bf16=False) as kv:
                rt.clear()
                attend(kv, n, pos0, n_head=n_head, n_kv=n_kv, head_dim=hd, causal=causal, window=window)
                names = [l["name"] for l in rt.launches()]
                assert any(kernel in m for m in names), (n_head, n_kv, hd, pos0, n, names)


@check
def scratch_that_a_graph_uses_outlives_larger_calls(rt, nh):
    """Warm up, capture, run a larger call: what the captured launches point to
    is still allocated, and given back with the cache. What was outgrown over
    many steps is together no longer than what is in use."""
    rows, dim = 4096, 512
    calls = {  # (BF16 cache, captured, larger)
        "staged X": (True, lambda kv: gemv(kv, "bf16", 16, 1024, 512), lambda kv: gemv(kv, "bf16", 1024, 1024, 512)),
        "K splits": (True, lambda kv: gemv(kv, "bf16", 16, 1024, 2560), lambda kv: gemv(kv, "bf16", 16, 8192, 2560)),
        "decode": (False, lambda kv: attend(kv, 1, 300), lambda kv: attend(kv, 16, 4000)),
        "long F32": (False, lambda kv: attend(kv, 1024), lambda kv: attend(kv, 2048)),
    }
    before = rt.lib.stub_live_bytes()
    for name, (bf16, small, large) in calls.items():
        with nh.KVCache([rows], [dim], bf16=bf16) as kv:
            small(kv)
            rt.clear()
            rt.capture(lambda: small(kv))
            held = {p for l in rt.launches() for p in l["scratch"]}
            left = {p: rt.left(p) for p in held}
            assert held and all(left.values()), name
            rt.clear()
            large(kv)
            assert held.isdisjoint(p for l in rt.launches() for p in l["scratch"]), f"{name}: the scratch did not grow"
            assert all(rt.left(p) == left[p] for p in held), name
        assert rt.lib.stub_live_bytes() == before, name
    with nh.KVCache([rows], [dim]) as kv:
        empty = rt.lib.stub_live_bytes()
        for n in range(2, 1025):
            rt.clear()
            gemv(kv, "bf16", n, 1024, 512)
        in_use = rt.left(rt.launches()[0]["xs"])
        assert in_use <= 2 * 1024 * 512 * 4 and rt.lib.stub_live_bytes() - empty < 2 * in_use


@pytest.mark.parametrize("name", sorted(CHECKS))
def test_host_path(stub, name):
    r = subprocess.run([sys.executable, str(HERE), str(stub), name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


if __name__ == "__main__":
    rt = Runtime(sys.argv[1])
    sys.path.insert(0, str(HERE.parents[1]))
    import libllmcpu_amd

    libllmcpu_amd.set_log_callback(lambda level, msg: None)
    CHECKS[sys.argv[2]](rt, libllmcpu_amd)
