#!/bin/bash
# Builds tensor_amd/lib/_otter_binding.so: the native per-call path of tensor_amd/capi.py (CPython + torch C++ API) over
# the C ABI of libotter_hip_int8.so. Plain g++: host code only.
set -e
cd "$(dirname "$0")"
mkdir -p ../lib
T=$(cd / && python3 -c "import importlib.util as u, os; print(os.path.dirname(u.find_spec('torch').origin))")
PY=$(cd / && python3 -c "import sysconfig; print(sysconfig.get_paths()['include'])")
g++ -std=c++17 -O2 -fPIC -shared -fvisibility=hidden -Wall -D__HIP_PLATFORM_AMD__=1 -DUSE_ROCM=1 -I"$PY" -isystem "$T/include" \
    -isystem "$T/include/torch/csrc/api/include" -isystem /opt/rocm/include binding.cpp -L"$T/lib" -lc10 -lc10_hip -ltorch_cpu \
    -ltorch_hip -ltorch_python -L../lib -lotter_hip_int8 -Wl,-rpath,'$ORIGIN' -Wl,-rpath,"$T/lib" -o ../lib/_otter_binding.so
echo "built $(cd ../lib && pwd)/_otter_binding.so"
