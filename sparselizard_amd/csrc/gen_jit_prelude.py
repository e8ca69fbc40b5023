"""Writes the source preludes of the kernels compiled at plan creation as C++
raw strings: include/slx.h, csrc/kernels/device.h and csrc/kernels/coef_device.h
for the coefficient and element kernels; the first two and csrc/kernels/tile.h
for the tile kernel, whose text (csrc/kernels/tile_jit.h) is a string of its own
(local includes, include guards and the C library headers, which the runtime
compiler does not ship, replaced by the fixed-width integer types).

usage: python3 gen_jit_prelude.py <output .inc>
"""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
KERNELS = os.path.join(HERE, "kernels")
SLX_H = os.path.join(HERE, "..", "..", "include", "slx.h")
STRINGS = [("kJitPrelude", True, [SLX_H, os.path.join(KERNELS, "device.h"), os.path.join(KERNELS, "coef_device.h")]),
           ("kTilePrelude", True, [SLX_H, os.path.join(KERNELS, "device.h"), os.path.join(KERNELS, "tile.h")]),
           ("kTileKernel", False, [os.path.join(KERNELS, "tile_jit.h")])]
TYPES = """#define SLX_RUNTIME_COMPILED
typedef signed char int8_t;
typedef unsigned char uint8_t;
typedef short int16_t;
typedef unsigned short uint16_t;
typedef int int32_t;
typedef unsigned int uint32_t;
typedef long int64_t;
typedef unsigned long uint64_t;
typedef __SIZE_TYPE__ size_t;
"""


def main():
    with open(sys.argv[1], "w") as fo:
        for name, types, files in STRINGS:
            out = [TYPES] if types else []
            for f in files:
                for line in open(f):
                    t = line.strip()
                    if t.startswith("#include") or t == "#pragma once":
                        continue
                    out.append(line)
            text = "".join(out)
            assert ')SLXJIT"' not in text
            fo.write('static const char %s[] = R"SLXJIT(' % name + text + ')SLXJIT";\n')


if __name__ == "__main__":
    main()
