"""The package's host side over a device runtime without a device (cpu_checks/host_hip.cc): only for processes started for
that, see run_case()."""
import ctypes
import importlib
import os
import subprocess
import sys
import tempfile
import types

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SOURCE = os.path.join(HERE, "cpu_checks", "host_hip.cc")


def build(directory):
    so = os.path.join(str(directory), "libhost_hip.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I/opt/rocm/include", SOURCE, "-o", so])
    return so


def run_case(so, test_file, name, *args, **env):
    """Runs function `name` of a test file in a process whose HIP calls go to the stand-in."""
    p = subprocess.run([sys.executable, os.path.abspath(test_file), so, name] + [str(a) for a in args], capture_output=True, text=True, timeout=100,
                       cwd=ROOT, env=dict(os.environ, **env))
    assert p.returncode == 0, p.stdout[-3000:] + p.stderr[-3000:]


def main(functions):
    host = Host(sys.argv[1])
    functions[sys.argv[2]](host, *sys.argv[3:])
    sys.stdout.flush()
    os._exit(0)  # (no destructors over the stand-in)


class Host:
    def __init__(self, so):
        self.hh = ctypes.CDLL(so, ctypes.RTLD_GLOBAL)  # before the library that calls it
        self.hh.hh_log.restype = ctypes.c_char_p
        # capi.py uses torch for its types' names only; torch itself would bring its device runtime along
        names = ("bool", "int8", "int16", "int32", "int64", "uint8", "float16", "float32", "float64")
        sys.modules["torch"] = types.SimpleNamespace(**{n: n for n in names})
        package = types.ModuleType("host_package")
        package.__path__ = [os.path.join(ROOT, "chainer-compiler_amd")]
        sys.modules["host_package"] = package
        self.capi = importlib.import_module("host_package.capi")
        self.chxvm = importlib.import_module("host_package.chxvm")
        self.lib = self.capi.lib()
        self.check(self.lib.chx_hip_init(0))

    def check(self, rc):
        assert rc == 0, self.lib.chx_hip_last_error()

    def log(self):
        return self.hh.hh_log().decode().splitlines()

    def launches(self):
        return [line[7:] for line in self.log() if line.startswith("launch ")]

    def clear(self):
        self.hh.hh_clear()

    def device_of(self, p):
        return self.hh.hh_device_of(ctypes.c_void_p(p))

    def malloc(self, nbytes):
        p = ctypes.c_void_p()
        self.check(self.lib.chx_hip_malloc(ctypes.byref(p), ctypes.c_size_t(nbytes)))
        return p.value

    def bytes(self, p, data):
        """`data` in device memory p (device memory is host memory here)."""
        ctypes.memmove(p, data, len(data))
        return p

    def stream(self):
        s = ctypes.c_void_p()
        self.check(self.lib.chx_hip_stream_create(ctypes.byref(s)))
        return s

    @staticmethod
    def dense(shape):
        strides = [1] * len(shape)
        for i in range(len(shape) - 2, -1, -1):
            strides[i] = strides[i + 1] * shape[i + 1]
        return strides

    def tensor(self, dtype, shape, strides=None, offset=0, base=None):
        """A descriptor; strides in elements (default dense), base: memory that is there already."""
        size = {"int8": 1, "uint8": 1, "float16": 2, "int32": 4, "float32": 4}[dtype]
        strides = self.dense(shape) if strides is None else strides
        span = 1 + sum((n - 1) * s for n, s in zip(shape, strides))
        base = base or self.malloc((span + offset) * size + 64)
        return self.capi.make_desc(base + offset * size, getattr(self.capi, dtype.upper()), shape, [s * size for s in strides])

    def channels_last(self, dtype, shape, pitch=None, offset=0):
        n, c, h, w = shape
        pitch = pitch or c
        return self.tensor(dtype, shape, [h * w * pitch, 1, w * pitch, pitch], offset)

    def plan(self, oc, c, k, pads=(0, 0), group=1):
        w, ws = self.tensor("int8", (oc, c, k, k)), self.tensor("float32", (oc,))
        zp, params = self.tensor("int8", (oc,)), self.capi.conv_params((1, 1), pads, pads, group)
        plan = ctypes.c_void_p()
        self.check(self.lib.chx_hip_qconv_plan_create(ctypes.byref(w), ctypes.byref(ws), ctypes.byref(zp), None, ctypes.byref(params), None, ctypes.byref(plan)))
        return plan

    def plan_run(self, plan, x, y, y_scale=0.05, y_zero_point=3, stream=None):
        return self.lib.chx_hip_qconv_plan_run(plan, ctypes.byref(x), ctypes.c_float(0.02), 128, ctypes.c_float(y_scale), y_zero_point, 0, ctypes.byref(y), stream)

    def program(self, builder):
        data, h = builder.serialize(), ctypes.c_void_p()
        rt = self.chxvm.runtime()
        assert rt.chxvm_program_create(data, len(data), ctypes.byref(h)) == 0, rt.chxvm_last_error()
        return h

    def run_fails(self, program, inputs):
        """What the runtime writes to stderr about a run that does not succeed."""
        rt, out = self.chxvm.runtime(), ctypes.c_void_p()
        with tempfile.TemporaryFile() as f:
            kept = os.dup(2)
            os.dup2(f.fileno(), 2)
            try:
                rc = rt.chxvm_program_run(program, *self.names_and(inputs), 0, ctypes.byref(out))
            finally:
                os.dup2(kept, 2)
                os.close(kept)
            assert rc != 0
            f.seek(0)
            return f.read().decode()

    def names_and(self, inputs):
        """{name: descriptor} as the C ABI takes it."""
        n = len(inputs)
        return (ctypes.c_char_p * n)(*[k.encode() for k in inputs]), (self.capi.Tensor * n)(*inputs.values()), n
