"""Which way a plan's tables go up, without a GPU: the library's plan calls over a stand-in for the runtime (tests/cpp/hip_stand_in.cpp),
loaded in front of it in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = """
import ctypes as C, sys
stand_in = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
current, memory_device, memory_type, stream, stream_device, at, batch = map(int, sys.argv[3:10])
i32, vp, z = C.c_int32, C.c_void_p, C.c_size_t
store = C.create_string_buffer((16 << 20) + 512)
base = (C.addressof(store) + 255) // 256 * 256
forms = []
for name in ("decode", "prefill"):
    create, plan, destroy = (getattr(lib, f"bz_{name}_plan{end}") for end in ("_create", "", "_destroy"))
    create.restype, destroy.argtypes = vp, [vp]
    h = create()
    stand_in.stand_in_set(current, memory_device, memory_type, stream_device)
    indptr = (i32 * (batch + 1))(*[4 * i for i in range(batch + 1)])
    if name == "decode":
        last = (i32 * batch)(*[16] * batch)
        plan.argtypes = [vp, vp, z, vp, z, vp, vp] + [C.c_uint32] * 6 + [vp]
        rc = plan(h, 1 << 40, 1 << 40, base + at, 16 << 20, indptr, last, batch, 8, 8, 128, 16, 0, stream)
    else:
        plan.argtypes = [vp, vp, z, vp, z, vp, vp] + [C.c_uint32] * 5 + [vp]
        rc = plan(h, None, 0, base + at, 16 << 20, indptr, indptr, batch, 8, 8, 128, 16, stream)
    forms.append((rc, stand_in.stand_in_kernels(), stand_in.stand_in_copies()))
    destroy(h)
print(forms)
"""
HOST, DEVICE, MANAGED, UNKNOWN = 1, 2, 3, -1  # (hipMemoryType; an address that the runtime does not know)


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stand_in") / "hip_stand_in.so")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-o", out,
                           os.path.join(ROOT, "tests", "cpp", "hip_stand_in.cpp")])
    return out


BY_KERNEL, BY_COPY = (0, 1, 0), (0, 0, 1)


@pytest.mark.parametrize("current,memory_device,memory_type,stream,stream_device,at,batch,form", [
    (0, 0, DEVICE, 0, 9, 0, 8, BY_KERNEL), (3, 3, DEVICE, 0, 9, 16, 8, BY_KERNEL), (3, 3, DEVICE, 2, 9, 0, 8, BY_KERNEL),
    (1, 1, DEVICE, 4096, 1, 0, 8, BY_KERNEL),
    (0, 1, DEVICE, 0, 9, 0, 8, BY_COPY),      # a workspace on another GPU than the current one
    (0, 1, DEVICE, 4096, 0, 0, 8, BY_COPY), (0, 0, DEVICE, 4096, 1, 0, 8, BY_COPY), (0, 1, DEVICE, 4096, 1, 0, 8, BY_COPY),
    (0, 0, HOST, 0, 9, 0, 8, BY_COPY), (0, 0, MANAGED, 0, 9, 0, 8, BY_COPY), (0, 0, UNKNOWN, 0, 9, 0, 8, BY_COPY),
    (0, 0, DEVICE, 0, 9, 8, 8, BY_COPY),      # inside a vector
    (0, 0, DEVICE, 0, 9, 0, 6000, BY_COPY),   # above half a megabyte
])
def test_a_kernel_writes_only_what_it_reaches(stand_in, current, memory_device, memory_type, stream, stream_device, at, batch, form):
    args = [current, memory_device, memory_type, stream, stream_device, at, batch]
    lib = os.path.join(ROOT, "blitz_scale_amd", "lib", "libbz_hip.so")
    out = subprocess.check_output([sys.executable, "-c", DRIVER, stand_in, lib, *map(str, args)], text=True)
    assert eval(out) == [form, form]
