"""What entry points of reinstinct_amd.runtime launch, without a GPU: `record(calls)` makes the calls in a child process on a
runtime that only writes launches down (fake_hip.c).  A call is (name, arguments) or ("option", [name, value]); pointers are
any aligned numbers.  A call's record is {"value": what it returned, "launches": [[kernel, grid, block, lds], ...]}."""
import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
P = 1 << 20                     # a pointer


def record(calls, tmp_path):
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    fake = str(tmp_path / "libamdhip64.so")
    subprocess.run([gcc, "-O1", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so", os.path.join(ROOT, "tests", "fake_hip.c"), "-o", fake], check=True)
    out = subprocess.run([sys.executable, os.path.abspath(__file__), fake], input=json.dumps(calls), capture_output=True, text=True, timeout=300,
                         cwd=ROOT)
    assert out.returncode == 0, out.stderr[-3000:]
    return json.loads(out.stdout)


def main():
    import ctypes
    fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)         # librein binds the runtime that is already there
    fake.fake_hip_record.restype = ctypes.c_char_p
    sys.path.insert(0, ROOT)
    from reinstinct_amd import _lib, runtime
    _lib.init()
    _lib.reset_options()
    done = []
    for name, args in json.load(sys.stdin):
        fake.fake_hip_clear()
        if name == "option":
            value = _lib.set_option(*args)
        elif name == "moe_ffn":
            value = runtime.moe_ffn(runtime.moe_shape(*args), P, P, P, P, P, P, P, P)
        else:
            value = getattr(runtime, name)(*args)
        launches = []
        for line in fake.fake_hip_record().decode().splitlines():
            kernel, *n = line.split()
            n = [int(v) for v in n]
            launches.append([kernel, n[:3], n[3], n[6]])
        done.append({"value": value, "launches": launches})
    json.dump(done, sys.stdout)


if __name__ == "__main__":
    main()
