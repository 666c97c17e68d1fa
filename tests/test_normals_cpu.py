"""Sine and cosine of the binary32 normals (sincos_turn in physics.h) against 64
bits, compiled for the host: no further off than sincospif, whose place they
take.  Bounds: sincospif's own errors over every word a draw can give, measured
on the device: largest 5.212e-8, root mean square 1.504e-8.

A turn u is reduced by a quarter exactly, so u = k 2^-27 up to 1/8 gives every
remainder that any u of a draw has; further u check the quadrants."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

PHYSICS = Path(__file__).resolve().parents[1] / "cmtj_amd" / "csrc" / "physics.h"

PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#define __device__
#define __forceinline__ inline
static uint32_t __float_as_uint(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
static float __uint_as_float(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
%s
static double worst = 0.0, sum = 0.0, n = 0.0;
static void at(float u, bool mean) {
  float s, c;
  sincos_turn(u, s, c);
  const double es = s - std::sin(2 * M_PI * (double)u), ec = c - std::cos(2 * M_PI * (double)u);
  worst = std::fmax(worst, std::fmax(std::fabs(es), std::fabs(ec)));
  if (mean) sum += es * es + ec * ec, n += 2;
}
int main() {
  for (uint32_t k = 1; k <= (1u << 24); ++k) at(std::ldexp((float)k, -27), false);
  uint64_t x = 88172645463325252ull;  // xorshift64
  for (int q = 0; q < (1 << 23); ++q) {
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    at(std::fma((float)(uint32_t)(x >> 32), 2.3283064365386963e-10f, 1.16415321826934814e-10f), true);
  }
  for (uint32_t o : {0u, 1u, 0xffffffffu, 0x1fffffffu, 0x20000000u, 0x40000000u, 0x80000000u, 0xc0000000u})
    at(std::fma((float)o, 2.3283064365386963e-10f, 1.16415321826934814e-10f), false);
  std::printf("%%.6e %%.6e\n", worst, std::sqrt(sum / n));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_sine_and_cosine_of_a_turn(tmp_path):
    text = PHYSICS.read_text()
    start = text.index("__device__ __forceinline__ void sincos_turn")
    body = text[start:text.index("\n}\n", start) + 3]
    src, exe = tmp_path / "turn.cpp", tmp_path / "turn"
    src.write_text(PROGRAM % body)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", str(src), "-o", str(exe)], check=True)
    worst, rms = map(float, subprocess.run([str(exe)], capture_output=True, text=True, check=True,
                                           timeout=120).stdout.split())
    print(f"[turn] largest error {worst:.4e}, rms {rms:.5e}")
    assert worst <= 5.212e-8 and rms <= 1.504e-8
