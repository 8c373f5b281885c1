"""What the library launches, seen on the CPU: each request runs in a process of its own
in which tests/fake_hip.cpp stands in for the HIP runtime."""
import ctypes
import json
import os
import pathlib
import re
import subprocess
import sys
import threading

ROOT = pathlib.Path(__file__).resolve().parents[1]


def build_fake(out_dir: pathlib.Path) -> pathlib.Path:
    lib = out_dir / "libfake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-o", str(lib),
                    str(ROOT / "tests" / "fake_hip.cpp")], check=True)
    return lib


def launches(fake: pathlib.Path, threads: list, env: dict | None = None) -> list:
    """``threads``: for each host thread its calls, ``[op, M, K, N, group, sms]`` with op
    "2_4", "w3", "meta3", "native", "noalloc" or "dense"; all on one stream, in step with
    each other where there are several.  Returns the launches in stream order as dicts:
    kernel, symbol (mangled, with its template arguments), grid, block, splits, thread;
    without the first call's clearing of the zero block."""
    req = json.dumps({"fake": str(fake), "threads": threads})
    out = subprocess.run([sys.executable, str(pathlib.Path(__file__)), req], capture_output=True, text=True,
                         cwd=ROOT, env={**os.environ, **(env or {})}, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    return json.loads(out.stdout.splitlines()[-1])


def _call(lib, op, M, K, N, g, sms):
    p, st = ctypes.c_void_p(4096), ctypes.c_void_p(64)  # operands and the stream: never dereferenced
    if op == "dense":
        return lib.marlin_hip_mul(p, p, p, p, M, N, K, p, g, 0, st, -1, -1, sms, 16)
    g = g // 2 if g != -1 else -1
    if op == "native":
        return lib.marlin_hip_mul_2_4_native(p, p, p, p, p, N, M, K, g, 0, st, sms)
    if op == "noalloc":
        return lib.marlin_hip_mul_2_4_noalloc(p, p, p, p, p, N, M, K, g, 0, st, -1, -1, sms)
    fn = getattr(lib, {"2_4": "marlin_hip_mul_2_4", "w3": "marlin_hip_mul_2_4_w3",
                       "meta3": "marlin_hip_mul_2_4_meta3"}[op])
    return fn(p, p, p, p, p, N, M, K, p, g, 0, st, -1, -1, sms, 16)


def _main(req):
    fake = ctypes.CDLL(req["fake"], mode=ctypes.RTLD_GLOBAL)
    fake.fake_hip_launch.restype = ctypes.c_char_p
    sys.path.insert(0, str(ROOT))
    from csed499ii_amd import _lib

    lib = _lib.load()
    start = threading.Barrier(len(req["threads"]))

    def work(i, calls):
        fake.fake_hip_caller(i)
        for call in calls:
            start.wait()
            err = _call(lib, *call)
            assert err == 0, (call, err, _lib.last_error())

    ts = [threading.Thread(target=work, args=a) for a in enumerate(req["threads"])]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    out = []
    u = [ctypes.c_uint(), ctypes.c_uint(), ctypes.c_int(), ctypes.c_int()]
    for i in range(fake.fake_hip_launches()):
        name = fake.fake_hip_launch(i, *map(ctypes.byref, u)).decode()
        if _base(name) != "fill_zero_kernel":
            out.append(dict(zip(("grid", "block", "splits", "thread"), (x.value for x in u)), kernel=_base(name),
                            symbol=name))
    print(json.dumps(out))


def _base(mangled: str) -> str:
    """_ZN4sm2415sm24_mid_kernelI... -> sm24_mid_kernel."""
    name, rest = mangled, mangled[3:]
    while m := re.match(r"\d+", rest):
        name, rest = rest[m.end():][:int(m.group())], rest[m.end() + int(m.group()):]
    return name


if __name__ == "__main__":
    _main(json.loads(sys.argv[1]))
