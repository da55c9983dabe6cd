// CPU emulation of the matrix-core kernels' step (mfma_step and
// mfma_step_residue) and of the short-tile batch kernel's runs
// (k_batch_short) against the oracle.
//
// The library's own tables (mrg8_amd/csrc/mrg8_math.hpp), lane by lane with
// the operand and result layouts of v_mfma_i32_16x16x32_i8 (lane l = n + 16 g
// holds K-group g of row/column n; result register i of lane l is row 4 g + i
// of column n).  A step's accumulators start from the step constants, class
// 2's doubled, and class 2's product is added twice; the residue comes from
// one two-term dot product of 16-bit halves.  A run of the batch kernel has
// eight tiles in sixteen columns, column n being half n / 8 of tile n mod 8,
// and ends with the product by A^128 that takes every column past the other
// half.  Every intermediate value is checked against the bound that the
// 32-bit arithmetic relies on.  Prints "mfma step emulation ok" and exits 0.
#include <cstdio>
#include <cstring>
#include <vector>

#include "mrg8_math.hpp"

extern "C" {
#include "mrg8_oracle.h"
}

using namespace mrg8;

namespace {

constexpr int kClasses = 4;
constexpr uint32_t kBeta = (1u << 27) + (1u << 19);
int failures = 0;

void check(bool ok, const char* what, long long a) {
  if (!ok && failures++ < 20) std::printf("FAIL %s (%lld)\n", what, a);
}

uint32_t digits(uint32_t w) { return (w + 0x40808080u) ^ 0x80808080u; }
int64_t digit(const uint32_t v[2], int i) { return (int8_t)((v[i / 4] >> (8 * (i % 4))) & 0xffu); }

typedef int64_t Acc[kClasses][16][16];  // [class][row][column]

void add_product(const std::vector<uint32_t>& A, const uint32_t B[64][2], int a, Acc C) {
  for (int m = 0; m < 16; ++m)
    for (int n = 0; n < 16; ++n)
      for (int g = 0; g < 4; ++g)
        for (int i = 0; i < 8; ++i) C[a][m][n] += digit(&A[((size_t)a * 64 + m + 16 * g) * 2], i) * digit(B[n + 16 * g], i);
}

uint32_t low_residue(uint64_t x) {
  check(x < 2ull * kP, "x range", (long long)x);
  return x < kP ? (uint32_t)x : (uint32_t)(x - kP);
}

// mfma_step_residue on accumulators that mfma_step left.
uint32_t step_residue(const Acc C, int m, int n) {
  for (int a = 0; a < kClasses; ++a) check(C[a][m][n] >= INT32_MIN && C[a][m][n] <= INT32_MAX, "accumulator", C[a][m][n]);
  const int64_t t = C[0][m][n] + 256 * C[1][m][n], u2 = C[2][m][n] + 512 * C[3][m][n];
  check(t >= 0 && t < 2 * (int64_t)kBeta + 65536, "t range", t);
  check(u2 >= 0 && u2 < 2 * (2 * (int64_t)kBeta + 32768) && u2 % 2 == 0, "2 u range", u2);
  const uint32_t t32 = (uint32_t)C[0][m][n] + ((uint32_t)C[1][m][n] << 8);
  const uint32_t u32 = (uint32_t)C[2][m][n] + ((uint32_t)C[3][m][n] << 9);
  check(t32 == t && u32 == u2, "32-bit combination", t);
  return low_residue((uint64_t)(u32 & 0xffffu) * (1u << 15) + (u32 >> 16) + t32);
}

// One step of sixteen columns: outputs 0..15 of each (as words), and the
// operands of the next step.
void step(const MfmaHostTables& mt, uint32_t B[64][2], uint32_t out[16][16]) {
  static Acc C;
  for (int a = 0; a < kClasses; ++a)
    for (int m = 0; m < 16; ++m)
      for (int n = 0; n < 16; ++n) C[a][m][n] = (int64_t)mt.c[((size_t)a * 4 + m / 4) * 4 + m % 4] * (a == 2 ? 2 : 1);
  for (int a : {0, 1, 2, 3, 2}) add_product(mt.a, B, a, C);
  for (int l = 0; l < 64; ++l) {
    const int n = l & 15, g = l >> 4;
    uint32_t r[4];
    for (int i = 0; i < 4; ++i) {
      r[i] = step_residue(C, 4 * g + i, n);
      out[n][mfma_position(g, i)] = r[i] + 1u;
    }
    for (int v = 0; v < 2; ++v) B[l][v] = digits(r[2 + v] + 1u);
  }
}

// The operands of every column multiplied by the stride tables' matrix.
void skip(const MfmaStrideTables& st, uint32_t B[64][2]) {
  static Acc C;
  std::memset(C, 0, sizeof C);
  for (int a = 0; a < kClasses; ++a) add_product(st.a, B, a, C);
  for (int l = 0; l < 64; ++l)
    for (int i = 0; i < 2; ++i) {
      const int n = l & 15, g = l >> 4, m = 4 * g + i;
      const int64_t t = C[0][m][n] + 256 * C[1][m][n], u = C[2][m][n] + 256 * C[3][m][n] + kBeta;
      const uint32_t k = st.k[(size_t)g * 2 + i];
      check(t + k >= 0 && t + k <= UINT32_MAX, "t + K range", t);
      check(u >= 0 && u <= 2 * (int64_t)kBeta, "skip u range", u);
      const uint64_t y = (uint64_t)u * 65536u + (uint64_t)(t + k);
      B[l][i] = digits(low_residue((y & kP) + (y >> 31)) + 1u);
    }
}

void operands(const uint32_t s[8], int n, uint32_t B[64][2]) {  // column n from the newest-first state s
  for (int g = 0; g < 4; ++g)
    for (int v = 0; v < 2; ++v) B[n + 16 * g][v] = digits(s[7 - (kMfmaWordOf[g] + v)]);
}

}  // namespace

int main() {
  MfmaHostTables mt;
  MfmaStrideTables st;
  const JumpTable jt;
  check(mfma_host_tables(16, 128, kClasses, kBeta, &mt), "step tables", 0);
  check(mfma_stride_tables(jt, 128, kClasses, kBeta, &st), "skip tables", 0);
  std::vector<uint32_t> tab((size_t)247 * 64);
  mrg8o_jump_table(tab.data());
  std::vector<std::vector<uint32_t>> states = {{kP, kP, kP, kP, kP, kP, kP, kP}, {0, 0, 0, 0, 0, 0, 0, 1},
                                               {kP, 0, 1, kP - 1, 0, kP, 2, 0}, {1, 1, 1, 1, 1, 1, 1, 1},
                                               {1, 0, 0, 0, 0, 0, 0, 0},        {0, kP, 0, kP, 0, kP, 0, kP}};
  uint64_t rng = 0x9e3779b97f4a7c15ull;
  while (states.size() < 64) {
    std::vector<uint32_t> v(8);
    for (auto& x : v) {
      rng ^= rng << 13, rng ^= rng >> 7, rng ^= rng << 17;
      x = (uint32_t)(rng % ((uint64_t)kP + 1));
    }
    states.push_back(v);
  }
  constexpr int kRuns = 3, kRun = 256;
  for (size_t first = 0; first < states.size(); first += 8) {  // a wave's eight tiles
    uint32_t B[64][2];
    std::vector<uint32_t> want[8];
    for (int tile = 0; tile < 8; ++tile) {
      uint32_t s[8];
      std::memcpy(s, states[first + tile].data(), sizeof s);
      operands(s, tile, B);
      mrg8o_jump(tab.data(), 128, s);
      operands(s, tile + 8, B);
      want[tile].resize(kRuns * kRun);
      std::memcpy(s, states[first + tile].data(), sizeof s);
      mrg8o_randint(s, want[tile].data(), want[tile].size());
    }
    for (int run = 0; run < kRuns; ++run) {
      for (int k = 0; k < 8; ++k) {
        uint32_t out[16][16];
        step(mt, B, out);
        for (int n = 0; n < 16; ++n)
          for (int o = 0; o < 16; ++o)
            check(out[n][o] == want[n % 8][(size_t)run * kRun + n / 8 * 128 + 16 * k + o], "output", 16 * k + o);
      }
      skip(st, B);
    }
  }
  if (failures) return std::printf("mfma step emulation: %d failures\n", failures), 1;
  std::printf("mfma step emulation ok: %zu tiles of %d outputs\n", states.size(), kRuns * kRun);
  return 0;
}
