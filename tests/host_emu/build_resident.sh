#!/bin/bash
# Host build of the resident RKC kernel (see resident_emu.cpp): the kernel's
# headers with their LDS declarations and the wait for outstanding stores put
# in the host's terms.  usage: build_resident.sh OUTDIR
set -euo pipefail
OUT=$1
HERE=$(cd "$(dirname "$0")" && pwd)
C=$(cd "$HERE/../../cerebellum-neuron-model-simulation-using-rkc_amd/csrc" && pwd)
mkdir -p "$OUT"
for f in detsum grid_mail rkc_resident; do
  sed -e 's/extern __shared__ double sm\[\];/double *const sm = emu_lds();/' \
      -e 's/__shared__ int s_late;/int \&s_late = *emu_late();/' \
      -e 's/__shared__ \(double\|long long\|int\) s_/static thread_local \1 s_/' \
      -e 's/asm volatile("s_waitcnt vmcnt(0)" ::: "memory");/__atomic_thread_fence(__ATOMIC_SEQ_CST);/' \
      "$C/$f.hpp" > "$OUT/$f.hpp"
done
g++ -std=c++17 -O1 -g -Wno-unknown-pragmas -DCB_HOST_EMU_HOST -ffp-contract=off -fPIC -shared -pthread -I "$HERE" -I "$OUT" -I "$C" \
  "$HERE/resident_emu.cpp" "$C/rkc_coef.cpp" -o "$OUT/libresident.so"
