#!/usr/bin/env bash
# Builds kernels/libternaspmm.so for MI355X (gfx950), the Python package's native host path and the tests/test_kernel harness.
# Run from anywhere:  bash kernels/compile.sh
# One hipcc compile per translation unit, all at once (each kernel family is instantiated in a
# file of its own), then one link.  -amdgpu-kernarg-preload-count: the first 16 dwords of a kernel's
# arguments arrive in scalar registers with the wave instead of being fetched by its first instructions
# (every launch of a decode step starts 0.05 - 0.3 us earlier).
set -euo pipefail
here="$(cd "$(dirname "${BASH_SOURCE[0]}")" && pwd)"
src="$here/../ternainfer_amd/csrc"
obj="$here/build"
mkdir -p "$obj"

flags=(-std=c++17 -O3 -fPIC --offload-arch=gfx950
       -Xclang -target-feature -Xclang -packed-fp32-ops
       -mllvm -amdgpu-kernarg-preload-count=16
       -Wall -Wno-unused-function)

pids=()
compile() {  # compile <source> <object> [extra flags]
    local s="$1" o="$2"; shift 2
    hipcc "${flags[@]}" "$@" -c "$src/$s" -o "$obj/$o" 2> >(grep -v "packed-fp32-ops' is not a recognized feature" >&2) &
    pids+=($!)
}
compile ternaspmm.hip ternaspmm.o
compile launch_reference.hip launch_reference.o
compile launch_decode_packed.hip launch_decode_packed.o
compile launch_prefill_packed.hip launch_prefill_packed_i8.o -DTERNA_PREFILL_ACT=int8_t -DTERNA_PREFILL_PRODUCERS
compile launch_prefill_packed.hip launch_prefill_packed_bf16.o -DTERNA_PREFILL_ACT=uint16_t
compile launch_mid.hip launch_mid.o
compile abi_fused.hip abi_fused.o
compile abi_chain.hip abi_chain.o
compile abi_attention.hip abi_attention.o
# the step's phases share no loop-invariant worth a register that one of them would then spill
compile abi_step.hip abi_step.o -mllvm -disable-machine-licm
compile launch_step_ordered.hip launch_step_ordered.o -mllvm -disable-machine-licm
# accumulators of the prompt-pass attention in ordinary vector registers (they are rescaled between matrix instructions)
compile abi_prefill_attention.hip abi_prefill_attention.o -mllvm -amdgpu-mfma-vgpr-form
compile abi_head.hip abi_head.o
compile abi_probe.hip abi_probe.o
compile format_host.cpp format_host.o
# The host path of the Python package: a CPython module on torch's C++ headers, bound to the library at run time.  The library
# itself needs neither; where they are missing it is all that is built, and the package says so when it is used.
native=
if torch="$(python3 -c 'import os, torch; print(os.path.dirname(torch.__file__))' 2> /dev/null)"; then
    python_include="$(python3 -c 'import sysconfig; print(sysconfig.get_paths()["include"])')"
    g++ -std=c++17 -O2 -fPIC -shared -Wall -Wno-unused-function -D__HIP_PLATFORM_AMD__=1 -DUSE_ROCM=1 \
        -isystem "$torch/include" -isystem "$torch/include/torch/csrc/api/include" -isystem "$python_include" -isystem /opt/rocm/include \
        "$src/py_native.cpp" -L"$torch/lib" -ltorch_python -ltorch_hip -ltorch_cpu -lc10 -lc10_hip -ldl -o "$here/../ternainfer_amd/_native.so" &
    native=$!
else
    echo "compile.sh: python3 has no PyTorch: the Python package's ternainfer_amd/_native.so is not built" >&2
fi
# every compile is waited for, also behind one that failed: none is left running
failed=0
for p in "${pids[@]}"; do wait "$p" || failed=1; done
native_failed=0
if [ -n "$native" ]; then wait "$native" || native_failed=1; fi
[ "$failed" = 0 ]

hipcc -shared -fPIC --offload-arch=gfx950 "$obj"/*.o -o "$here/libternaspmm.so"

if [ -f "$here/../tests/test_kernel.hip" ]; then
    hipcc -std=c++17 -O2 --offload-arch=gfx950 \
        "$here/../tests/test_kernel.hip" \
        -L"$here" -lternaspmm -lhipblas \
        -Wl,-rpath,'$ORIGIN/../kernels' \
        -o "$here/../tests/test_kernel"
fi
[ "$native_failed" = 0 ]
