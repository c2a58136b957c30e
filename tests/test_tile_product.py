"""The large tiles' product (csrc/tile_product.h) as far as it shows without a GPU: the offsets of its loads, worked out by the
kernels' own functions, and the order in which the compiler leaves the first ones."""

import re
import shutil
import subprocess

import pytest

from fastgen_amd.kernels import _lib

PROGRAM = r"""
#include "tile_product.h"
#include <cstdio>
#include <vector>
typedef unsigned long long u64;
static long long loads = 0;
static int failed = 0;
static void need(bool ok, const char* what, int a, int b, int c, int d, int e) {
  if (!ok && failed++ < 20) printf("%s: %d %d %d %d %d\n", what, a, b, c, d, e);
}
// Whether 16 bytes at a lane's offset are read: the scalar offset no part of the check, taken off the size without and with
// wrapping, added to the lane's.
static void ways(const TileLoad& l, unsigned lane, bool (&reads)[4]) {
  reads[0] = (u64)lane + 16 <= l.bytes;
  reads[1] = (u64)lane + l.at + 16 <= l.bytes;
  reads[2] = l.bytes && (u64)lane + 16 <= (unsigned)(l.bytes - l.at);
  reads[3] = (u64)(unsigned)(lane + l.at) + 16 <= l.bytes;
}
// `there`: it has to be read; `zeros`: it has to be zeros; and whatever is read lies in [0, size) behind `base`.  (That a size of 0 does
// not wrap is seen on the GPU, where the rows of x have NaN behind them.)
static void check(const TileLoad& l, unsigned lane, u64 base, u64 size, bool there, bool zeros, const char* what, int a, int b, int c, int d, int e) {
  bool reads[4];
  ways(l, lane, reads);
  ++loads;
  for (bool r : reads) {
    need(r || !there, what, a, b, c, d, e);
    need(!r || !zeros, what, a, b, c, d, e);
    need(!r || base + lane + l.at + 16 <= size, what, a, b, c, d, e);
  }
}
template <int MB, int NB, int NST, int WS, bool ONE>
static void tile(int N, int K, int splits, bool two) {  // two: the experts' gate and up, 8 NB columns of either a wave
  typedef TileProduct<MB, NB, NST, WS, ONE> P;
  static const char matrix[1] = {0};
  const int width = two ? 8 * NB : 16 * NB, blocks = (N + 15) / 16, steps = (K / 64 + splits - 1) / splits;
  TileOperands op;
  op.w_row = (unsigned)K * 32u;
  const u64 size = (u64)blocks * op.w_row;
  for (int n0 = 0; n0 < N + 4 * width; n0 += width) {
    for (int part = 0; part < 2; ++part) op.set_w(part, matrix, n0 / 16 + (part && !two ? P::HALF : 0), blocks, part ? NB - P::HALF : P::HALF);
    for (int first = 0; first < K / 64; first += steps) {
      const int n_stages = min(steps, K / 64 - first), last = (n_stages + P::U - 1) / P::U * P::U;
      for (int nb = 0; nb < NB; ++nb)
        for (int t = 0; t < 2 * last + WS - 1; ++t) {
          const int part = nb < P::HALF ? 0 : 1, block = n0 / 16 + (two && part ? nb - P::HALF : nb);
          const bool stage = t < 2 * n_stages, there = stage && block < blocks;
          for (unsigned lane : {0u, 63u * 16}) {
            const TileLoad l = P::w_load(op, nb, t, first, n_stages);
            const u64 base = (const char*)op.w[part] - matrix;
            check(l, lane, base, size, there, !stage, "W", MB * 1000 + NB, N, K, n0, t);
            if (there) need(base + l.at == (u64)block * op.w_row + 1024u * (2 * first + t), "W's place", NB, N, K, n0, t);
          }
        }
    }
  }
}
template <int MB, int NB, int NST, int WS, bool ONE>
static void rows(long long ldx, int K, int n_rows) {  // of x, at most n_rows of a tile there
  typedef TileProduct<MB, NB, NST, WS, ONE> P;
  TileOperands op;
  op.x_bytes = 2u * (unsigned)((n_rows - 1) * ldx + K);
  const int n = K / 64, last = (n + P::U - 1) / P::U * P::U + P::LA;
  for (int row = 0; row < 16 * MB; ++row)
    for (unsigned chunk : {0u, 112u})
      for (int s : {0, n / 2, n - 1, n, last - 1}) {
        const unsigned lane = op.row_offset(row < n_rows, row, (int)ldx, chunk);
        const bool there = row < n_rows && s < n;
        const TileLoad l = P::x_load(op, s, 0, n);
        check(l, lane, 0, op.x_bytes, there, !there, "x", MB, n_rows, K, row, s);
        if (there) need((u64)lane + l.at == 2ull * row * ldx + 128 * s + chunk, "x's place", MB, n_rows, K, row, s);
      }
}
template <int MB, int NB, int NST, int WS, bool ONE>
static void all(bool moe) {
  for (int N : {1, 8, 16, 17, 33, 48, 63, 65, 112, 129, 200, 257, 272, 515, 1040})
    for (int K : {64, 128, 192, 320, 704})
      for (int splits : {1, 2, 3})
        if ((K / 64 + splits - 1) / splits * (splits - 1) < K / 64) tile<MB, NB, NST, WS, ONE>(N, K, splits, false), moe ? tile<MB, NB, NST, WS, ONE>(N, K, splits, true) : void();
  for (int n_rows : {1, 7, 16 * MB - 1, 16 * MB}) {
    rows<MB, NB, NST, WS, ONE>(64, 64, n_rows);
    rows<MB, NB, NST, WS, ONE>(776, 704, n_rows);
    rows<MB, NB, NST, WS, ONE>(7812496, 2048, n_rows);           // the widest rows there may be (512 of them and one row's k: 4e9 bytes)
    if (MB <= 8) rows<MB, NB, NST, WS, ONE>(7690000, 7689984 / 64 * 64, n_rows);  // and the longest k with them
  }
}
int main() {
  all<16, 4, 5, 4, true>(false), all<16, 3, 5, 4, true>(false), all<8, 4, 5, 4, false>(true), all<8, 3, 5, 4, false>(false);
  all<8, 2, 5, 8, false>(true), all<4, 2, 5, 8, false>(true), all<16, 4, 5, 8, true>(true), all<8, 4, 5, 8, true>(true);
  all<4, 4, 5, 8, true>(true), all<4, 4, 5, 4, false>(true);
  printf("%lld loads, %d wrong\n", loads, failed);
  return failed != 0;
}
"""


@pytest.fixture(scope="module")
def hipcc():
    try:
        path = _lib._hipcc()
    except Exception:
        path = None
    if not path or not (shutil.which(path)):
        pytest.skip("no compiler")
    return path


def test_loads_stay_inside_whichever_way_the_scalar_offset_is_checked(hipcc, tmp_path):
    """A buffer load is checked against its buffer's size; whether its scalar offset takes part in that, and how, must not
    matter: what is not there is zeros where zeros are needed and never a read behind the matrix or the rows."""
    (tmp_path / "loads.cpp").write_text(PROGRAM)
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", f"-I{_lib.CSRC}", str(tmp_path / "loads.cpp"), "-o",
                    str(tmp_path / "loads")], check=True, timeout=120)
    run = subprocess.run([str(tmp_path / "loads")], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout


def first_loads(listing):
    """The buffer loads in front of a product's first barrier, one string per product: x to LDS, W to registers, as they lie
    in the listing."""
    found, here = [], ""
    for line in listing.splitlines():
        if "s_barrier" in line and len(here) > 8:  # in a product there are fewer between two matrix instructions
            found.append(here)
        if "v_mfma" in line or "s_barrier" in line:
            here = ""
        elif "buffer_load_dwordx4" in line:
            here += "x" if re.search(r"\blds\b", line) else "W"
    return found


@pytest.mark.parametrize("source", ["gemm_large", "moe"])
def test_first_loads_are_in_the_order_that_the_wait_counts(hipcc, tmp_path, source):
    """The wait in front of a product's first barrier lets a number of loads be on their way: it is right only if all of x was
    asked for before the first of W."""
    flags = [f for f in _lib.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "-S", "--offload-device-only", f"-I{_lib.CSRC}", str(_lib.CSRC / f"{source}.hip"), "-o",
                    str(tmp_path / "listing")], check=True, capture_output=True, timeout=300)
    n_products = 0
    for name, body in re.findall(r"^(_Z\d+(?:gemm|moe)_large_kernel\w+):(.*?)^\.Lfunc_end", (tmp_path / "listing").read_text(), re.S | re.M):
        mb, nb, nst, ws = (int(n) for n in re.findall(r"Li(\d+)E", name)[:4])
        # (a loop's last load may lie in front of the next product's; one of the product's own would be missing behind)
        products = [p.lstrip("W") for p in first_loads(body)]
        # tiles of 256 rows also go in halves; the experts' as products of 64 rows on
        rows = [m for m in (16, 8, 4) if m == mb or (m < mb and (source == "moe" or m == 8))]
        assert sorted(products) == sorted("x" * ((nst - 2) * m // 2) + "W" * ((ws - 1) * nb) for m in rows), name
        n_products += len(products)
    assert n_products >= 14
    assert first_loads("buffer_load_dwordx4 v1, s[0:3], 0 offen lds\n" * 4 + "buffer_load_dwordx4 v[0:3], v1, s[0:3], 0 offen\n" * 5
                       + "buffer_load_dwordx4 v1, s[0:3], 0 offen lds\n" * 2 + "s_barrier\n") == ["xxxxWWWWWxx"]
