"""The canonical row units (xs_units.h) read nothing past a row's last word where the rows are in global memory: the last
row of the last expert ends where the arena ends, and the next byte may lie in no allocation.  The header is compiled
for the host, with the device's names defined, and each format's row is put right before a page that faults."""
import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "xestrata-win_amd" / "csrc"

DEVICE = r"""
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#include <initializer_list>
#define __device__
#define __host__
#define __constant__
#define __forceinline__ inline
struct alignas(8) uint2 { uint32_t x, y; };
struct alignas(16) uint4 { uint32_t x, y, z, w; };
namespace xs {
constexpr int kQ8_0 = 8, kQ4_K = 12, kQ6_K = 14, kIQ4_XS = 23;
inline float h2f(uint16_t h) { return (float)h / 1024.0f; }
inline int sdot4(int a, int b, int c) {
    for (int i = 0; i < 4; ++i) c += (int)(int8_t)(a >> (8 * i)) * (int)(int8_t)(b >> (8 * i));
    return c;
}
inline int table16_lookup(uint32_t i, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return (int)(i * 0x01010101u ^ a ^ b ^ c ^ d);
}
inline uint32_t host_alignbyte(uint32_t hi, uint32_t lo, uint32_t n) {
    return (uint32_t)((((uint64_t)hi << 32) | lo) >> (8 * (n & 3)));
}
}
#define __builtin_amdgcn_alignbyte xs::host_alignbyte
"""

MAIN = r"""
#include "xs_units.h"
#include <cstdio>
#include <cstdlib>
#include <sys/mman.h>
using namespace xs;
static int8_t q[4096];
static float d8[128];
static int us16[256];

// the same `blocks` blocks once with room after them and once right before the page that faults
template <int T, bool S256, bool GLOBAL>
int rows(int values, int bytes, int blocks, uint8_t* end) {
    static uint8_t roomy[16384] __attribute__((aligned(16)));
    const int n = blocks * bytes, pad = (16 - n % 16) % 16;   // (a row starts on 16 bytes or, of two, follows another)
    for (int i = 0; i < n; ++i) roomy[pad + i] = (uint8_t)rand();
    uint8_t* const last = end - n - pad;
    memcpy(last, roomy, pad + n);
    const Act a[1] = {Act{q, d8, us16}};
    const int units = blocks * values / Unit<T, S256>::kUnit;
    for (int u = 0; u < units; ++u) {
        float x[1] = {0.0f}, y[1] = {0.0f};
        Unit<T, S256>::template apply<1, false>(roomy, pad, u, a, 1, x);
        Unit<T, S256>::template apply<1, GLOBAL>(last, pad, u, a, 1, y);
        if (memcmp(x, y, 4)) return printf("type %d unit %d: %g %g\n", T, u, x[0], y[0]), 1;
    }
    return 0;
}

int main(int argc, char** argv) {
    uint8_t* const m = (uint8_t*)mmap(nullptr, 1 << 16, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    uint8_t* const end = m + (1 << 15);
    if (mprotect(end, 1 << 15, PROT_NONE)) return 2;
    for (auto& v : q) v = (int8_t)rand();
    for (auto& v : d8) v = (float)(rand() % 100) / 64.0f;
    for (auto& v : us16) v = rand() % 4000 - 2000;
    if (argc > 1) return rows<kQ8_0, false, false>(32, 34, 8, end);   // LDS reads, off the end
    int bad = 0;
    for (int blocks : {1, 2, 3, 8, 16}) {
        bad |= rows<kQ8_0, false, true>(32, 34, blocks, end) | rows<kQ8_0, true, true>(32, 34, blocks, end);
        bad |= rows<kQ4_K, false, true>(256, 144, blocks, end) | rows<kQ4_K, true, true>(256, 144, blocks, end);
        bad |= rows<kQ6_K, false, true>(256, 210, blocks, end) | rows<kQ6_K, true, true>(256, 210, blocks, end);
        bad |= rows<kIQ4_XS, false, true>(256, 136, blocks, end) | rows<kIQ4_XS, true, true>(256, 136, blocks, end);
    }
    return bad;
}
"""


def test_global_rows_stay_inside_the_arena(tmp_path):
    (tmp_path / "xs_units.h").write_text((CSRC / "xs_units.h").read_text())
    (tmp_path / "xs_device.h").write_text(DEVICE)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "rows"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-I", str(tmp_path), "-o", str(exe), str(tmp_path / "main.cpp")],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout)
    # the form for rows in LDS does read the word after a Q8_0 row, so the page after it tells the two apart
    assert subprocess.run([str(exe), "lds"], capture_output=True).returncode < 0


def test_direct_rows_take_the_global_form():
    """The kernels that read rows from the blob itself ask for that form: the persistent layer's direct instances and the
    one-token kernel's waiters."""
    fused, t1 = ((CSRC / f).read_text() for f in ("decode_fused.hip", "decode_t1.hip"))
    assert fused.count("apply<NE, DIRECT>(rb,") == 1 and fused.count("apply<M, DIRECT>(rb,") == 1
    assert t1.count("apply<1, true>(row,") == 1
