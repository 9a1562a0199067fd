#!/bin/bash
# Builds libobme_hip.so for gfx950 in-tree (next to this script's package):
# each translation unit is compiled to an object in parallel, then linked.
# Packed FP32 instructions are disabled (-packed-fp32-ops).
set -euo pipefail
HERE="$(cd "$(dirname "${BASH_SOURCE[0]}")" && pwd)"
OUT="${OBME_OUT:-${HERE}/../oceanbiome/libobme_hip.so}"
HIPCC="${HIPCC:-/opt/rocm/bin/hipcc}"
FLAGS=(--offload-arch=gfx950 -O3 -std=c++17 -fPIC
       -Xclang -target-feature -Xclang -packed-fp32-ops
       -Wall -Wno-unused-function -Wno-unused-variable -Wno-pass-failed)
TMP="$(mktemp -d)"
trap 'rm -rf "${TMP}"' EXIT
# obme_pisces.hip: FP32 division and square root need not be correctly
# rounded (its FP32 arithmetic is the FP32-mixed path; FP64 is unaffected).
pids=()
objs=()
compile() {  # object source flags...
    objs+=("${TMP}/$1.o")
    "${HIPCC}" "${FLAGS[@]}" "${@:3}" ${OBME_EXTRA_FLAGS:-} -c -o "${TMP}/$1.o" "${HERE}/$2.hip" &
    pids+=($!)
}
# the sweep and the wave kernels: one object per model (NPZD, LOBSTER) and set
# of its components (1 the carbonate system, 2 oxygen)
for mc in "2 3" "2 1" "2 2" "2 0" "1 2" "1 0"; do
    read -r m c <<< "${mc}"
    compile "obme_sweep_${m}_${c}" obme_sweep "-DOBME_TU_MODEL=${m}" "-DOBME_TU_CARB=${c}"
    compile "obme_wave_${m}_${c}" obme_wave "-DOBME_TU_MODEL=${m}" "-DOBME_TU_CARB=${c}"
done
compile obme_pisces obme_pisces -fno-hip-fp32-correctly-rounded-divide-sqrt
compile obme_api obme_api
for p in "${pids[@]}"; do wait "$p"; done
"${HIPCC}" --offload-arch=gfx950 -fPIC -shared -o "${OUT}.tmp" "${objs[@]}"
mv "${OUT}.tmp" "${OUT}"
echo "built ${OUT}"
