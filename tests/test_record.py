"""The short way into the C ABI (csrc/lng_record.cpp) against the way through ctypes: the same calls, for plain arguments and
for everything that is not plain, end in the same launches with the same arguments, the same errors and the same texts. On the
null device, in a process of its own (a process binds one library)."""
import os
import subprocess
import sys
import sysconfig

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "loadngo_amd", "csrc")

PROGRAM = r"""
import ctypes, sys
import numpy as np
from loadngo_amd import compute as C
C.LIB_PATH = sys.argv[1]
lib = C.library()
short = C._record
assert short is not None
lib.lng_null_launch_count.restype = ctypes.c_size_t
lib.lng_null_launch.argtypes = [ctypes.c_size_t, ctypes.POINTER(ctypes.c_char_p), ctypes.POINTER(ctypes.c_uint * 3), ctypes.POINTER(ctypes.c_uint * 3),
                                ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(ctypes.c_size_t)]

class Other(C.Slice):
    __slots__ = ()

class Count(int):
    pass

S = C.Slice
half = C.Slice(0, 0, 4)
del half.len
gpu = C.Gpu(0)
bufs = [gpu.buffer(1 << 20) for _ in range(8)]
weights = gpu.resident(np.zeros(1 << 20, np.uint8))

def launches():
    out = []
    for i in range(lib.lng_null_launch_count()):
        name, grid, block, args, size = ctypes.c_char_p(), (ctypes.c_uint * 3)(), (ctypes.c_uint * 3)(), ctypes.c_void_p(), ctypes.c_size_t()
        assert lib.lng_null_launch(i, ctypes.byref(name), ctypes.byref(grid), ctypes.byref(block), ctypes.byref(args), ctypes.byref(size)) == 0
        out.append((name.value, list(grid), list(block), ctypes.string_at(args.value, size.value)))
    return out

def attempt(f):
    lib.lng_null_clear()
    b = gpu.batch(bufs)
    b.attach(weights)
    try:
        f(b)
        recorded = b.dispatches()
        done = b.run()
        return recorded, done.gpu_time, launches()
    except Exception as e:
        return type(e).__name__, str(e)
    finally:
        b.drop()

def both(f):
    C._record = short
    first = attempt(f)
    C._record = None
    second = attempt(f)
    C._record = short
    return first, second

shape = lambda t=1, window=C.FULL, scale=0.125, slots=64: C.GroupedShape(t, 40, 8, 2, 64, window, slots, scale)
qs, kv, out = S(0, 0, 8 * 64 * 4), S(1, 0, 41 * 2 * 64 * 4), S(2, 0, 8 * 64 * 4)
tq, tkv, tout = S(0, 0, 32 * 8 * 64 * 4), S(1, 0, 96 * 2 * 64 * 4), S(2, 0, 32 * 8 * 64 * 4)
sinks = S(3, 0, 32)
m = (S(8, 0, 64 * 64), S(8, 8192, 64 * 2 * 2))
many = [(m, S(4, 0, 256), 64), (m, S(5, 0, 256), 64)]
item = C.decode_items([C.DecodeItem(0, 0, 0, 0, None, 40, C.FULL, 64), C.DecodeItem(2048, 2048, 0, 0, 0, 9, 4, 64)])
fresh = C.prepare_items([C.PrepareItem(n=1, start=3, slots=64)])
where = dict(q=0, k=1, v=2, table=3, q_out=4, k_cache=5, v_cache=6)
bias = S(8, 0, 8 * 64 * 4)
odd = [3, 0, -1, 2**64, 2**64 - 1, True, 1.0, None, "1", np.int64(1), np.float32(0.5), Count(1), half, Other(0, 0, 2048)]
slices = [S(0, 0, 2048), Other(0, 0, 2048), S(np.int64(0), 0, 2048), S(0, True, 2048), S(0, -1, 2048), S(0, 0, 2**64), S(0, 0.0, 2048), S(9, 0, 2048),
          S(0, 0, 2044), half, None, (0, 0, 2048), 7]

calls = []
def vary(f, *args):
    # the call as it is, and with each argument replaced by each odd one (and by each slice where it is one)
    calls.append(lambda b: f(b, *args))
    for i, a in enumerate(args):
        for other in (slices if isinstance(a, C.Slice) else odd):
            calls.append(lambda b, i=i, other=other: f(b, *args[:i], other, *args[i + 1:]))

B = C.Batch
vary(B.attention_grouped, qs, kv, S(3, 0, kv.len), out, shape(), C.F32)
vary(B.attention_grouped_with_sinks, (qs, kv, S(4, 0, kv.len)), sinks, out, shape(), C.F32)
vary(B.attention_grouped_tiled, tq, tkv, S(4, 0, tkv.len), tout, shape(32, slots=96), C.F32)
vary(B.attention_grouped_tiled_with_sinks, [tq, tkv, S(4, 0, tkv.len)], sinks, tout, shape(32, slots=96), C.F32)
vary(B.copy_rows, (S(0, 0, 512), 32), (S(1, 0, 512), 32), 4, 32, C.F32, None)
vary(B.copy_rows, [S(0, 0, 512), 32], (S(1, 0, 256), 32), 4, 32, C.F32, C.BF16)
vary(B.attention_decode_batched, 0, 1, 2, 3, 4, item, 8, 2, 64, 0.125, C.F32)
vary(B.attention_decode_batched, 0, 1, 2, 3, 4, [C.DecodeItem(0, 0, 0, 0, None, 40, C.FULL, 64)], 8, 2, 64, 1, C.F32)
vary(B.attention_decode_batched, 0, 1, 2, 3, 4, fresh, 8, 2, 64, 0.125, C.F32)
vary(B.rmsnorm_rows, (S(0, 0, 1024), S(1, 0, 256)), 4, (64, 64), 1e-5)
vary(B.add_rows, S(0, 0, 1024), (S(1, 0, 1024), 64), 4, 64)
vary(B.prepare_attention, where, fresh, 8, 2, 64, 64, C.BF16, None, None, None)
vary(B.prepare_attention, where, fresh, 8, 2, 64, None, C.F32, bias, S(8, 0, 512), S(8, 0, 512))
vary(B.prepare_attention, {k: v for k, v in where.items() if k != "table"}, fresh, 8, 2, 64)
vary(B.prepare_attention, dict(where, q=np.int64(0)), [C.PrepareItem(n=1, start=3, slots=64)], 8, 2, 64)
for f in (B.gemm_q8_0, B.gemm_q8_0_bf16):
    vary(f, m, S(1, 0, (256 if f is B.gemm_q8_0 else 128) * 2), S(2, 0, 512), 64, 64, 2, (64, 64))
vary(B.gemm_q8_0_tiled, m, S(1, 0, 256 * 32), S(2, 0, 256 * 32), 64, 64, 32, [64, 64])
vary(B.gemm_q8_0_many, many, S(1, 0, 256), 64, 1, 64)
vary(B.gemm_q8_0_many, tuple(many), S(1, 0, 256), 64, 1, 64)
vary(B.gemm_q8_0_many, many * 3, S(1, 0, 256), 64, 1, 64)
vary(B.gemm_q8_0_many, [(m, S(4, 0, 256))], S(1, 0, 256), 64, 1, 64)
vary(B.gemm_q8_0_many_normed, many, S(1, 0, 256), (S(8, 0, 256), 1e-5), 64, 1, 64)
vary(B.gemm_q8_0_many_normed, many, S(1, 0, 256), (S(8, 0, 256), 1), 64, 1, 64)
vary(B.gemm_q8_0_residual, m, S(1, 0, 256), S(8, 0, 256), S(2, 0, 256), 64, 64, 1, (64, 64), C.F32)
vary(B.gemm_q8_0_residual, m, S(1, 0, 128), None, S(2, 0, 256), 64, 64, 1, (64, 64), C.BF16)

worked = 0
for n, f in enumerate(calls):
    first, second = both(f)
    assert first == second, (n, first, second)
    worked += len(first) == 3
assert worked > 40, worked

# batches: buffers given twice, freed, resident, of the other kind; a batch dropped twice, run twice, used after it ran
def batches(buffers):
    try:
        b = gpu.batch(buffers)
        b.drop(); b.drop()
        return "made"
    except Exception as e:
        return type(e).__name__, str(e)
gone = gpu.buffer(64)
gone.free()
for buffers in ([], bufs, bufs + bufs[:1], [weights], [gone], [gpu.buffer(64) for _ in range(70)]):
    C._record = short
    first = batches(buffers)
    C._record = None
    assert batches(buffers) == first, buffers
for way in (short, None):
    C._record = way
    b = gpu.batch(bufs)
    b.add_rows(S(0, 0, 1024), (S(1, 0, 1024), 64), 4, 64)
    for f in (b.wait, lambda: b.run().gpu_time, b.run, lambda: b.add_rows(S(0, 0, 1024), (S(1, 0, 1024), 64), 4, 64)):
        try:
            print(f())
        except Exception as e:
            print(type(e).__name__, e)
    seen = []
    b.drop()
    c = gpu.batch(bufs)
    c.commit(lambda done: seen.append(done.gpu_time))
    c.wait()
    assert len(seen) == 1 and isinstance(seen[0], float)
    c.drop()
    for f in (c.wait, c.commit):
        try:
            print(f())
        except Exception as e:
            print(type(e).__name__, e)
    print("--")
print(len(calls), "calls,", worked, "made")
"""


def test_the_short_way_and_ctypes_make_the_same_calls(tmp_path):
    from loadngo_amd import compute as C
    assert C._record is not None, "csrc/lng_record.cpp is not built"
    lib = str(tmp_path / "null.so")
    null = os.path.join(CSRC, "null_device")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-pthread", "-DLNG_NULL_DEVICE", "-I" + null, os.path.join(CSRC, "lng_hip.cpp"),
                           os.path.join(null, "null_hip.cpp"), "-o", lib])
    run = subprocess.run([sys.executable, "-c", PROGRAM, lib], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert run.returncode == 0, run.stdout[-4000:]
    first, second, _ = run.stdout.split("--\n")
    assert first == second, run.stdout


def test_the_extension_is_named_for_the_python_it_was_built_for(tmp_path, monkeypatch):
    """One without a tag would be imported by any Python, whatever its objects look like."""
    from loadngo_amd import build
    (tmp_path / "_record.so").write_bytes(b"of an older build")
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    made = build.build_record()
    assert [p.name for p in tmp_path.iterdir()] == ["_record" + sysconfig.get_config_var("EXT_SUFFIX")] == [os.path.basename(made)]
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})  # without headers: none, and none left
    assert build.build_record() is None and list(tmp_path.iterdir()) == []
