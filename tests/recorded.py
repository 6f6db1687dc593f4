"""Calls of libmythos_oil.so with its HIP runtime replaced by
hip_recorder.c: what each call launches, allocates and returns, without a GPU.

As a program (a process of its own, so that torch's HIP runtime is not
loaded): reads a JSON list of calls from stdin, each {"fn", "args", and
optionally "capture": the stream that is capturing}, and prints a JSON list of
{"rc", "kernels": [[name, grid]], "mallocs", "bytes", "error"}.  As a module:
`run(calls)` does that, `library()` loads both libraries into this process.
"""
import ctypes as C
import json
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.environ.get("MYTHOS_OIL_LIB") or os.path.join(ROOT, "mythos.cpp_amd", "libmythos_oil.so")
P, I64, F32 = C.c_void_p, C.c_int64, C.c_float
SIG = {
    "mth_oil8_gemv": [P, P, P, P, I64, I64, I64, P],
    "mth_oil4_gemv": [P, P, I64, P, P, I64, I64, I64, P],
    "mth_oil4_gemv_noalloc": [P, P, I64, P, P, I64, I64, I64, P],
    "mth_oil4_gemm_prefill": [P, P, P, I64, P, I64, I64, I64, P],
    "mth_i2s_gemv": [P, F32, P, P, P, I64, I64, I64, P],
    "mth_i2s_gemv_f32": [P, F32, P, P, I64, I64, I64, P],
    "mth_i2s_gemm": [P, P, P, I64, I64, I64, P],
    "mth_attention_decode": [P, P, P, P, I64, I64, I64, I64, I64, I64, P],
    "mth_argmax": [P, P, I64, I64, P],
    "mth_workspace_reserve": [I64, P],
}


def library():
    """(recorder, library) in this process."""
    d = tempfile.mkdtemp()
    so = os.path.join(d, "hip_recorder.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-o", so,
                    os.path.join(ROOT, "tests", "hip_recorder.c")], check=True)
    rec = C.CDLL(so, mode=C.RTLD_GLOBAL)
    os.remove(so)
    os.rmdir(d)
    rec.rec_name.restype = C.c_char_p
    rec.rec_grid.restype = C.c_uint32
    rec.rec_malloc_bytes.restype = C.c_uint64
    rec.rec_capture.argtypes = rec.rec_hold.argtypes = [P]
    lib = C.CDLL(LIB)
    for n, a in SIG.items():
        getattr(lib, n).argtypes, getattr(lib, n).restype = a, C.c_int
    lib.mth_last_error.restype = C.c_char_p
    return rec, lib


def main():
    rec, lib = library()
    out = []
    for c in json.load(sys.stdin):
        rec.rec_reset()
        if c.get("capture") is not None:
            rec.rec_capture(c["capture"])
        rc = getattr(lib, c["fn"])(*c["args"])
        out.append({"rc": rc, "mallocs": rec.rec_mallocs(), "bytes": rec.rec_malloc_bytes(),
                    "error": lib.mth_last_error().decode(),
                    "kernels": [[rec.rec_name(i).decode(), [rec.rec_grid(i, d) for d in range(3)]]
                                for i in range(rec.rec_launches())]})
    print(json.dumps(out))


def child(args, text=None):
    r = subprocess.run([sys.executable, *args], input=text, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return r.stdout


def run(calls):
    return json.loads(child([os.path.abspath(__file__)], json.dumps(calls)))


if __name__ == "__main__":
    main()
