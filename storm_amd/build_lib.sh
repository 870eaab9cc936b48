#!/bin/sh
# Builds the gfx950 engine library storm_amd/_lib/libstorm_amd.so.  Fails if a
# transport kernel spills vector registers (check_registers.py).
set -e
here=$(cd "$(dirname "$0")" && pwd)
mkdir -p "$here/_lib"
if ! /opt/rocm/bin/hipcc --offload-arch=gfx950 -O3 -std=c++17 -fPIC -shared \
  -ffp-contract=off -Xclang -target-feature -Xclang -packed-fp32-ops \
  -Rpass-analysis=kernel-resource-usage \
  -I"$here/../include" \
  -o "$here/_lib/libstorm_amd.so.tmp" "$here/csrc/engine.hip" 2> "$here/_lib/remarks.txt.tmp"; then
  cat "$here/_lib/remarks.txt.tmp" >&2
  exit 1
fi
mv "$here/_lib/remarks.txt.tmp" "$here/_lib/remarks.txt"
grep "warning:" "$here/_lib/remarks.txt" >&2 || true
python3 "$here/check_registers.py" "$here/_lib/remarks.txt"
mv "$here/_lib/libstorm_amd.so.tmp" "$here/_lib/libstorm_amd.so"
