"""Load offsets of the FP8 prefill kernels (ling-engine_amd/csrc/lq_prefill_offsets.hpp), compiled here for the host.
A raw buffer load is out of range where vector offset >= bytes - scalar offset; for every lane, load and K block that a
kernel issues, those past the operand's rows and blocks among them, the scalar offset has to stay within the operand (the
difference never goes below zero), a load inside has to read its own bytes, and a load outside has to be out of range (the
256 x 256 tile's last of too few rows reads others that exist)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ling-engine_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include "lq_prefill_offsets.hpp"
using namespace lq;
static long long tests = 0, bad = 0;
static void expect(bool inside, unsigned v, unsigned s, unsigned width, unsigned bytes, unsigned want, const char* what,
                   int a, int b, bool any = false) {
  ++tests;
  const unsigned long long at = static_cast<unsigned long long>(v) + s;
  const bool ok = s <= bytes && (inside ? at == want && want + width <= bytes
                                        : v >= bytes - s || (any && at + width <= bytes));
  if (!ok && bad++ < 5) std::printf("%s: rows %d, row %d: v %u s %u of %u\n", what, a, b, v, s, bytes);
}
// where unit u of row n, block kb, lies: 16-row tiles of KB blocks of 2048 bytes, rows 8h + g, K pieces 32t + 16q
static unsigned weight_at(int n, int u, int kb, int KB) {
  const int h = (n % 16) / 8, g = n % 8, q = u / 4, t = u % 4;
  return ((n / 16) * KB + kb) * 2048u + (((h * 2 + q) * 8 + g) * 4 + t) * 16u;
}

// the smaller tiles: loads of TN weight rows, TM tokens and their scales, blocks 0 .. KB - 1 + stages
static void tile(int TN, int TM, int stages, int M, int N, int KB) {
  const int K = KB * 128;
  const unsigned wb = static_cast<unsigned>(N) * K, xb = static_cast<unsigned>(M) * K, sb = static_cast<unsigned>(M) * KB * 4;
  for (int kb = 0; kb < KB + stages; ++kb) {
    const unsigned past = kb < KB ? 0u : kLoadNothing;
    for (int n0 = 0; n0 < N; n0 += TN)
      for (int n = n0; n < n0 + TN; ++n)
        for (int u = 0; u < 8; ++u)
          expect(n < N && kb < KB, (n < N ? weight_unit_offset(n, u, KB) : kLoadNothing) | past, block_offset(kb, KB, 2048), 16,
                 wb, weight_at(n, u, kb, KB), "tile weights", N, n);
    for (int m0 = 0; m0 < M; m0 += TM)
      for (int m = m0; m < m0 + TM; ++m) {
        for (int u = 0; u < 8; ++u)
          expect(m < M && kb < KB, (m < M ? activation_unit_offset(m, u, K) : kLoadNothing) | past, block_offset(kb, KB, 128),
                 16, xb, static_cast<unsigned>(m * K + kb * 128 + u * 16), "tile activations", M, m);
        expect(m < M && kb < KB, (m < M ? static_cast<unsigned>(m * KB * 4) : kLoadNothing) | past, block_offset(kb, KB, 4), 4,
               sb, static_cast<unsigned>((m * KB + kb) * 4), "tile scales", M, m);
      }
  }
}

// the 256 x 256 tile: loads i = 0 .. 3 64 rows apart, over the rows that are there or not
static void whole(int M, int N, int KB) {
  const int K = KB * 128;
  const unsigned wb = static_cast<unsigned>(N) * K, xb = static_cast<unsigned>(M) * K;
  for (int kb = 0; kb < KB; ++kb)
    for (int i = 0; i < 4; ++i)
      for (int row = 0; row < 64; ++row)
        for (int u = 0; u < 8; ++u) {
          for (int n0 = 0; n0 < N; n0 += 256) {
            const int n = n0 + row + 64 * i;
            expect(n < N, weight_unit_offset(n0 + row, u, KB), kb * 2048u + i * 64u * K, 16, wb, weight_at(n, u, kb, KB),
                   "weights", N, n);
          }
          for (int m0 = 0; m0 < M; m0 += 256) {
            const int m = m0 + row + 64 * i;
            const unsigned s = kb * 128u + (i < 3 ? i * 64u * K : last_load_offset(M, 64u * K));
            expect(m < M, activation_unit_offset(m0 + row, u, K), s, 16, xb, static_cast<unsigned>(m * K + kb * 128 + u * 16),
                   "activations", M, m, i == 3 && M < 193);
          }
        }
}

int main() {
  static_assert(kWholeRows == 129, "the fewest rows that whole() is checked with");
  const int ms[] = {1, 2, 3, 5, 63, 64, 65, 129, 200}, ns[] = {128, 256, 384}, kbs[] = {1, 2, 3, 5, 9};
  const int shapes[][3] = {{64, 64, 4}, {128, 64, 3}, {128, 128, 4}, {128, 128, 2}};
  for (int M : ms)
    for (int N : ns)
      for (int KB : kbs)
        for (auto& s : shapes) tile(s[0], s[1], s[2], M, N, KB);
  const int whole_ms[] = {129, 130, 160, 192, 193, 200, 256, 300, 449, 512}, whole_ns[] = {256, 384, 640};
  for (int M : whole_ms)
    for (int N : whole_ns)
      for (int KB : kbs) whole(M, N, KB);
  std::printf("tests %lld bad %lld\n", tests, bad);
  return bad != 0 || tests < 100000;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_scalar_offsets_stay_within_the_operand(tmp_path):
    src = tmp_path / "offsets.cpp"
    exe = tmp_path / "offsets"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
