#!/usr/bin/env bash
# Builds qtensor/libqtensor_hip.so for gfx950 (cross-compiles without a GPU) and qtensor/_direct.so, the native host side
# of a quantize or dequantize call (plain C++ against torch's headers).
# Sources compile in parallel to objects under csrc/build/, then link.
set -euo pipefail
here="$(cd "$(dirname "${BASH_SOURCE[0]}")" && pwd)"
out="${QT_OUT:-${here}/../qtensor/libqtensor_hip.so}"
obj="${QT_OBJ:-${here}/build}"
HIPCC="${HIPCC:-/opt/rocm/bin/hipcc}"
# -ffp-contract=off: the nearest-entry rule needs two separately rounded fp32 subtractions.
# packed-fp32-ops is switched off for the device pass: some packed forms give wrong results now and then.
FLAGS=(-O3 -std=c++17 --offload-arch=gfx950 -fPIC -ffp-contract=off -fno-fast-math
       -Xclang -target-feature -Xclang -packed-fp32-ops
       -Wall -Wno-unused-command-line-argument -I"${here}" -I"${here}/../../include")
mkdir -p "${obj}"
pids=()
objs=()
for src in "${here}"/qt_*.hip; do
  o="${obj}/$(basename "${src%.hip}").o"
  objs+=("${o}")
  "${HIPCC}" "${FLAGS[@]}" "$@" -c "${src}" -o "${o}" &
  pids+=($!)
done
# Beside the library that it is bound to (none for a library built somewhere else), and from scratch: what is there may be of
# another torch.  The library does without it, so it is no reason not to link the library.
build_direct() {
  local to="${here}/../qtensor/_direct.so" where
  rm -f "${to}"
  where="$("${PYTHON:-python3}" -c 'import os, sysconfig, torch; print(os.path.dirname(torch.__file__), sysconfig.get_paths()["include"], torch.__version__, sep="\n")')" || return 1
  mapfile -t where <<< "${where}"
  "${CXX:-g++}" -O2 -std=c++17 -shared -fPIC -Wall -D__HIP_PLATFORM_AMD__=1 -DUSE_ROCM=1 -DQT_TORCH_VERSION="\"${where[2]}\"" \
    -I"${where[0]}/include" -I"${where[0]}/include/torch/csrc/api/include" -I"${HIP_PATH:-/opt/rocm}/include" -I"${where[1]}" \
    "${here}/direct_call.cpp" -o "${obj}/_direct.so" \
    -L"${where[0]}/lib" -lc10 -lc10_hip -ltorch_cpu -ltorch_hip -ltorch -ltorch_python -Wl,-rpath,"${where[0]}/lib" || return 1
  mv "${obj}/_direct.so" "${to}"
}
direct=""
if [[ -z "${QT_OUT:-}" ]]; then
  build_direct &
  direct=$!
fi
for p in "${pids[@]}"; do wait "${p}"; done
"${HIPCC}" --offload-arch=gfx950 -shared -fPIC "${objs[@]}" -o "${out}"
echo "built ${out}"
if [[ -n "${direct}" ]] && ! wait "${direct}"; then
  echo "warning: qtensor/_direct.so was not built; quantize and dequantize calls have their host side in Python" >&2
fi
