"""Plans are looked up per device: what a layer is cut into depends on the device's compute units and shader clock, and a process
may launch on several.  The library runs against a stand-in for the two runtime calls that it asks about devices, in which device
1 has another clock than device 0."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DEVICES = r"""
#include <hip/hip_runtime_api.h>
static int current;
void set_device(int d) { current = d; }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t what, int d)
{
    if (what == hipDeviceAttributeClockRate)
        *v = d ? 600000 : 2400000;
    else if (what == hipDeviceAttributeMultiprocessorCount)
        *v = 256;
    else if (what == hipDeviceAttributeMaxSharedMemoryPerBlock)
        *v = 163840;
    else
        return hipErrorInvalidValue;
    return hipSuccess;
}
"""

# prints [[device, plans of every layer], ...] for the devices given, asked in that order in one process
CHILD = r"""
import ctypes, importlib.util, json, random, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
spec = importlib.util.spec_from_file_location("binding", sys.argv[2])
binding = importlib.util.module_from_spec(spec)
spec.loader.exec_module(binding)
lib = binding.load()

rng = random.Random(3)
layers = []
for _ in range(150):
    d = binding.ConvDesc()
    k, s, c, co = rng.choice((1, 3, 5)), rng.choice((1, 1, 2)), rng.randint(3, 500), rng.randint(8, 600)
    h = rng.randint(k, 60)
    d.input_shape[:], d.filter_shape[:] = (rng.randint(1, 64), h, rng.randint(k, 60), c), (k, k, c, co)
    d.strides[:], d.dilations[:] = (1, s, s, 1), (1, 1, 1, 1)
    d.padding, d.data_format, d.num_bits = binding.PAD_SAME, binding.FORMAT_NHWC, 8
    layers.append(d)

out = []
for device in json.loads(sys.argv[3]):
    shim.set_device(device)
    info = [ctypes.c_int() for _ in range(3)]
    assert lib.axc_device_info(*map(ctypes.byref, info)) == 0
    assert info[2].value == (600000 if device else 2400000), info[2].value
    plans = []
    for d in layers:
        plan, nbytes = (ctypes.c_int32 * 8)(), ctypes.c_size_t()
        assert lib.axc_conv2d_workspace_bytes(ctypes.byref(d), ctypes.byref(nbytes)) == 0
        row = [nbytes.value]
        for call in (lib.axc_conv2d_tile_plan, lib.axc_conv2d_matrix_plan, lambda d, p: lib.axc_conv2d_direct_plan(d, 0, p)):
            assert call(ctypes.byref(d), plan) == 0
            row += list(plan)
        plans.append(row)
    out.append([device, plans])
print(json.dumps(out))
"""


def test_each_device_has_its_own_plans(pkg, tmp_path):
    shim, source = tmp_path / "libdevices.so", tmp_path / "devices.c"
    source.write_text(DEVICES)
    subprocess.run(["gcc", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(source), "-o", str(shim)],
                   check=True)

    def plans(*devices):
        got = subprocess.run([sys.executable, "-c", CHILD, str(shim), os.path.join(ROOT, "tf-approximate_amd", "_lib.py"),
                              json.dumps(devices)], check=True, stdout=subprocess.PIPE, text=True)
        return [p for _, p in json.loads(got.stdout)]

    (first,), (second,) = plans(0), plans(1)
    assert sum(a != b for a, b in zip(first, second)) >= 3     # the clock decides some of them
    assert plans(0, 1, 0) == [first, second, first]
    assert plans(1, 0) == [second, first]
