"""The kernel launches that calls of the operation library make, without a
GPU: python launches.py RECORDER.so reads a JSON list of calls
[name, arguments] from its input and prints each call's result and launches.
An argument {"conv": [...]} is a convolution descriptor and "p" a distinct
device address, which is never read."""
import ctypes as C
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


class Launch(C.Structure):
    _fields_ = [("kernel", C.c_void_p), ("grid", C.c_uint * 3), ("block", C.c_uint * 3),
                ("lds", C.c_size_t), ("lds_limit", C.c_int)]


def main(recorder):
    rec = C.CDLL(recorder, mode=C.RTLD_GLOBAL)
    rec.rec_launch.restype = C.POINTER(Launch)
    sys.path.insert(0, os.path.join(os.path.dirname(HERE), "aet-cnn_amd"))
    import aetcnn
    ops, out, keep = aetcnn.ops(), [], []
    for name, args in json.load(sys.stdin):
        rec.rec_reset()
        a = []
        for i, v in enumerate(args):
            if isinstance(v, dict):
                keep.append(aetcnn.ConvDesc(*v["conv"]))
                v = C.byref(keep[-1])
            a.append((i + 1) << 32 if v == "p" else v)
        rc = getattr(ops, name)(*a)
        ls = [rec.rec_launch(i)[0] for i in range(rec.rec_count())]
        out.append(dict(rc=rc, launches=[
            dict(kernel=v.kernel, grid=list(v.grid), block=list(v.block), lds=v.lds,
                 lds_limit=v.lds_limit) for v in ls]))
    json.dump(out, sys.stdout)


def record(calls, tmp_path):
    so = os.path.join(str(tmp_path), "recorder.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so,
                    os.path.join(HERE, "launch_recorder.c")], check=True)
    r = subprocess.run([sys.executable, os.path.join(HERE, "launches.py"), so],
                       input=json.dumps(calls), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout)


if __name__ == "__main__":
    main(sys.argv[1])
