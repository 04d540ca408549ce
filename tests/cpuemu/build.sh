#!/bin/bash
# Host build of the library for AddressSanitizer checks: the HIP sources are
# compiled as C++ against tests/cpuemu/hip/hip_runtime.h, which runs every GPU
# thread of a workgroup as a host thread (workgroups one after another).
# -fsanitize=bounds also checks every index into a fixed-size array member,
# which ASan cannot: kernel arguments are structs passed by value, and their
# copies sit in stack memory without redzones.
#   tests/cpuemu/build.sh OUT.so
set -e
D=$(cd "$(dirname "$0")"; pwd)
R=$(cd "$D/../.."; pwd)
C=$R/specfempp_amd/csrc
OUT=$1
T=$(mktemp -d)
FLAGS="-std=c++20 -g -O1 -fPIC -fsanitize=address,bounds -fno-sanitize-recover=bounds -fno-omit-frame-pointer -I$D -I$C -I$R/include"
# the 3-D block path is refused on the device but built and checked here
grep -q 'run->scatter == SFX_SCATTER_BLOCK && !host_only' "$C/engine.hip"
sed 's/run->scatter == SFX_SCATTER_BLOCK && !host_only/false/' "$C/engine.hip" > "$T/engine.hip"
g++ $FLAGS -x c++ -c "$T/engine.hip" -o "$T/engine.o" &
for f in batch block3d kernels acoustic general3d patch2d; do
  g++ $FLAGS -x c++ -c "$C/$f.hip" -o "$T/$f.o" &
done
g++ $FLAGS -c "$C/assembly.cpp" -o "$T/assembly.o" &
g++ $FLAGS -c "$C/patch2d.cpp" -o "$T/patch2d_host.o" &
wait
g++ -shared -fsanitize=address,bounds -o "$OUT" "$T"/engine.o "$T"/batch.o "$T"/kernels.o "$T"/acoustic.o "$T"/general3d.o "$T"/block3d.o "$T"/patch2d.o "$T"/patch2d_host.o "$T"/assembly.o -lpthread
rm -rf "$T"
