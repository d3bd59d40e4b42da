"""Host-side rules of the library, compiled from its own headers with the host compiler and run on the CPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "tessera_amd" / "csrc"


def _run(tmp_path, source, *args):
    """Compiles one program against the library's headers and returns what it printed."""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-pthread", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True, timeout=60).stdout


def test_few_row_offsets_stay_in_32_bits(tmp_path):
    """Few-row products off the 16-byte grid: wherever the rule admits one, the largest offsets that the kernel's
    lanes form lie inside the buffer range (A) and inside 32 bits (B); ordinary sizes are admitted."""
    cases = _few_row_cases()
    out = _run(tmp_path, r"""
#include "few_rows.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  for (int i = 1; i + 4 < argc; i += 5)
    std::printf("%d\n", tsr950::few_rows16_in_range(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), atol(argv[i + 3]), atol(argv[i + 4])));
}
""", *[x for c in cases for x in c])
    got = [bool(int(x)) for x in out.split()]
    assert len(got) == len(cases)
    for (m, n, k, lda, ldb), ok in zip(cases, got):
        pitch = max(lda, -(-k // 8) * 8)
        # lane (row m - 1, upper half) of A's second load in a slice; row 31 and the last column of B's slice
        a_last = (m - 1) * pitch * 2 + 16 + 32 + 15
        b_last = (31 * ldb + n - 1) * 2 + 1
        assert not ok or (a_last < 2 ** 31 - 1 and b_last < 2 ** 32), (m, n, k)
        if max(lda, k) <= 1 << 24 and ldb <= 1 << 25:
            assert ok, (m, n, k)                          # nothing of the ordinary range is turned away
    assert not got[0] and not got[1] and got[2]


def _few_row_cases():
    cases = [(64, 8, 17_100_000), (1, 1 << 26, 32), (64, 50257, 4100)]
    cases += [(m, n, k) for m in (1, 2, 9, 32, 33, 64) for n in (8, 9, 1003, 1 << 24, 69_273_000, 69_274_000, 1 << 28)
              for k in (1, 33, 4097, 1 << 24, 17_043_000, 17_044_000, 34_600_000, 1 << 30, 2 ** 31 - 1)]
    return [(m, n, k, k, n) for m, n, k in cases] + [(3, 100, 64, 1 << 29, 104), (3, 100, 64, 64, 1 << 27)]


def test_8bit_streaming_splits_count_their_partials(tmp_path):
    """K splits of the 8-bit streaming kernel at shapes whose forced splits were timed (11.8 us in 16 parts against 14.2 in
    32, and so on): within a few per cent of the best, never past one workgroup per compute unit or one slice a wave."""
    timed = {(64, 1024, 8192): (12, 16), (48, 512, 14336): (16, 32), (32, 2048, 8192): (8, 12), (64, 2048, 4096): (6, 8),
             (48, 1280, 5120): (8, 16), (16, 8192, 8192): (4, 4), (32, 4096, 14336): (8, 8), (16, 3072, 8192): (8, 10),
             (64, 8192, 8192): (4, 4), (16, 14336, 4096): (1, 2), (32, 8192, 2048): (1, 3)}
    tiled = [(16, 128256, 2048), (32, 128256, 2048)]         # timed 7 to 11 % below the streaming kernel
    timed |= {(64, 28672, 4096): (1, 1), (48, 4096, 4096): (4, 8)}
    many = [(m, n, k) for m in (1, 32, 33, 64) for n in (16, 129, 4096, 33000, 1 << 24) for k in (16, 63, 1024, 8193, 1 << 23)]
    out = _run(tmp_path, r"""
#include "gemm8_schedule.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3) {
    const int M = atoi(argv[i]), N = atoi(argv[i + 1]), K = atoi(argv[i + 2]), w = tsr950::gemm8_skinny_waves(M, K, false);
    std::printf("%d %d %d\n", tsr950::gemm8_skinny_splits(w, M, N, K), w, tsr950::select_gemm8_schedule(M, N, K).skinny);
  }
}
""", *[x for c in [*timed, *tiled, *many] for x in c])
    got = [tuple(map(int, line.split())) for line in out.splitlines()]
    for (shape, (low, high)), (splits, _, skinny) in zip(timed.items(), got):
        assert low <= splits <= high and skinny, (shape, splits)
    assert not any(skinny for _, _, skinny in got[len(timed):len(timed) + len(tiled)])
    for (m, n, k), (splits, waves, _) in zip(many, got[len(timed) + len(tiled):]):
        strips = -(-n // 128)
        assert waves == (8 if m <= 32 else 4) and 1 <= splits and (splits == 1 or (splits * strips <= 256 and splits * waves * 64 <= k))


def test_padded_decode_fills_whole_rounds(tmp_path):
    """Key splits and route of decode at padded head dimensions, at shapes timed both ways: one workgroup per compute unit
    at DP 128 and 256, two at 64."""
    splits = {(128, 256, 500): 1, (128, 192, 1000): 1, (128, 64, 2048): 4, (128, 128, 2048): 2, (64, 256, 500): 1, (64, 256, 4096): 2,
              (128, 512, 4096): 1, (256, 256, 250): 1, (256, 64, 300): 2, (128, 8, 64): 1}
    general = {(256, 500, 80): 0, (257, 500, 80): 1, (512, 64, 96): 1, (512, 1024, 80): 0, (768, 500, 80): 0, (1024, 250, 112): 1,
               (512, 500, 48): 0, (512, 500, 64): 0, (512, 500, 128): 0, (512, 500, 160): 0}
    out = _run(tmp_path, r"""
#include "attn_rules.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  for (int i = 2; i + 2 < argc; i += 3) {
    const int a = atoi(argv[i]), b = atoi(argv[i + 1]), c = atoi(argv[i + 2]);
    std::printf("%d\n", i < 2 + 3 * atoi(argv[1]) ? tsr950::pad_splits(a, b, (c + 31) / 32, a == 256 ? 2 : 4) : (int)tsr950::pad_general(a, b, c));
  }
}
""", len(splits), *[x for c in [*splits, *general] for x in c])
    got = dict(zip([*splits, *general], map(int, out.split())))
    assert got == {**splits, **general}


def test_attention_shapes_follow_their_timings(tmp_path):
    """Waves and key splits of the plain attention forward at shapes timed both ways (causal, D 128 where not said)."""
    wide, four = 8, 4
    timed = {  # (B, Hq, Hkv, Sq, Sk, D, causal): waves
        (2, 32, 8, 500, 500, 128, 1): four, (1, 32, 8, 1000, 1000, 128, 1): four, (1, 32, 8, 2048, 2048, 128, 1): four,
        (9, 32, 8, 384, 384, 128, 1): four, (1, 32, 8, 4096, 4096, 128, 1): wide, (4, 32, 8, 4096, 4096, 128, 1): wide,
        # few rows on long contexts, the 8-wave form with its own splits: 282 us against 298, 517 / 540, 548 / 587, 287 / 318
        (1, 32, 8, 512, 32768, 128, 1): wide, (1, 32, 8, 1024, 32768, 128, 1): wide, (1, 32, 8, 256, 131072, 128, 1): wide,
        (1, 8, 8, 1024, 65536, 128, 1): wide, (1, 32, 8, 512, 4096, 128, 1): four, (1, 32, 8, 256, 16384, 128, 1): four,
        (2, 16, 16, 233, 1133, 80, 1): four, (1, 32, 8, 227, 1127, 80, 1): four, (7, 8, 1, 108, 1008, 64, 1): wide,
        # one round of 8 waves, a half-empty second block: 17.5 / 18.5; a small third one 17.2 / 16.3
        (4, 32, 4, 350, 350, 128, 1): wide, (8, 16, 16, 384, 384, 128, 1): wide, (4, 32, 4, 300, 300, 128, 1): four,
        # heads that share no K and V, past the caches: 39.3 / 46.0, 59.6 / 66.9; within them 35.4 / 34.0; half as wide 23.2 / 21.6
        (16, 32, 32, 256, 256, 128, 1): wide, (24, 32, 32, 256, 256, 128, 1): wide, (10, 32, 32, 256, 256, 128, 1): four,
        (16, 32, 32, 256, 256, 64, 1): four, (20, 32, 32, 500, 500, 128, 1): wide, (24, 32, 32, 640, 640, 128, 1): four,
        (18, 8, 8, 1559, 1559, 80, 1): four, (1, 8, 8, 256, 65536, 128, 1): four,
        (16, 8, 8, 1572, 1572, 128, 1): four, (34, 32, 32, 107, 307, 80, 1): four, (26, 32, 32, 99, 999, 128, 1): four,
        (1, 8, 2, 3065, 3065, 80, 1): four, (1, 32, 4, 342, 342, 80, 1): wide, (41, 8, 8, 881, 881, 80, 1): four,
        (1, 8, 1, 180, 1080, 128, 1): wide, (1, 16, 16, 133, 1033, 128, 1): wide, (8, 16, 16, 160, 160, 128, 1): four,
        (1, 8, 1, 3333, 4233, 80, 1): wide, (10, 8, 2, 640, 640, 80, 1): wide, (10, 8, 2, 512, 512, 80, 1): four, (8, 16, 16, 300, 300, 80, 1): wide}
    out = _run(tmp_path, r"""
#include "attn_rules.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  for (int i = 1; i + 6 < argc; i += 7) {
    int v[7];
    for (int j = 0; j < 7; ++j) v[j] = atoi(argv[i + j]);
    const tsr950::FlashProblem p{v[0], v[1], v[2], v[3], v[4], v[5], false};
    const int off = p.Sk > p.Sq ? p.Sk - p.Sq : 0;
    const auto f = tsr950::flash_shape(p, [&](int q0, int rows) { return ((v[6] ? std::min(p.Sk, q0 + rows + off) : p.Sk) + 63) / 64; });
    std::printf("%d %d %d\n", f.waves, f.nsplit, tsr950::flash_blocks_last(p));
  }
}
""", *[x for c in timed for x in c])
    for (shape, waves), line in zip(timed.items(), out.splitlines()):
        got, nsplit, last = map(int, line.split())
        b, hq, hkv, sq, sk, d, _ = shape
        assert got == waves, (shape, line)
        assert nsplit == 1 or (b * hq * -(-sq // 256) < 192 and nsplit <= -(-sk // 64) // 8)
        assert last == (hq != hkv or d <= 96 or b * hkv < 300 or 4 * d * b * hkv * sk < 9e7)


# A device of 100 units, counted, in the place of HIP: `used` units are out, `syncs` synchronisations happened.
_FAKE_DEVICE = r"""
#include "device_pool.h"
#include <cstdio>
#include <cstdlib>
using namespace tsr950;
static const size_t kUnit = size_t(64) << 20;
static size_t used = 0, syncs = 0;
static std::map<void*, size_t> out;
static char* next_address = reinterpret_cast<char*>(4096);
struct Fake {
  static bool device(int* d) { *d = 0; return true; }
  static PoolAlloc malloc(void** p, size_t bytes) {
    if (used + bytes > 100 * kUnit) return PoolAlloc::kNoMemory;
    *p = next_address; next_address += bytes; used += bytes; out[*p] = bytes;
    return PoolAlloc::kOk;
  }
  static bool free(void* p) { used -= out.at(p); out.erase(p); return true; }
  static bool synchronize(int dev) { ++syncs; return dev == 0; }
};
static DevicePool<Fake> pool;
static void check(bool ok, int line) { if (!ok) { std::printf("line %d\n", line); std::exit(1); } }
#define CHECK(x) check(x, __LINE__)
"""


def test_pool_gives_its_blocks_to_other_allocations(tmp_path):
    """A full device: an allocation outside the pool (a stream's workspace, a raw buffer, a stream-ordered temporary)
    takes what the pool has cached, and fails only where the memory is really out."""
    out = _run(tmp_path, _FAKE_DEVICE + r"""
int main() {
  void *a, *b, *p = nullptr;
  CHECK(pool.malloc(&a, 20 * kUnit) && pool.malloc(&b, 20 * kUnit));
  CHECK(pool.free(a, false) == PoolStatus::kOk && pool.free(b, true) == PoolStatus::kOk && used == 40 * kUnit);
  CHECK(pool.free(a, false) == PoolStatus::kForeign);
  auto take = [&](size_t units) { return pool.allocate([&] { return Fake::malloc(&p, units * kUnit); }); };
  CHECK(take(60) && used == 100 * kUnit);                // fits beside the cached blocks: they stay
  CHECK(take(30) && used == 90 * kUnit);                 // 40 were idle in the pool
  CHECK(!take(30) && used == 90 * kUnit);                // nothing cached any more
  CHECK(take(10));
  CHECK(!pool.malloc(&a, kUnit));
  int calls = 0;                                         // another error is not answered by a second attempt
  CHECK(!pool.allocate([&] { ++calls; return PoolAlloc::kFailed; }) && calls == 1);
  std::printf("ok\n");
}
""")
    assert out == "ok\n"


def test_pool_blocks_settle_behind_their_last_owner(tmp_path):
    """A block handed out again at once has its last owner's work queued on it: `settle` waits for the device then, and
    only then."""
    out = _run(tmp_path, _FAKE_DEVICE + r"""
int main() {
  void *a, *b, *c;
  CHECK(pool.malloc(&a, kUnit) && pool.settle(a) == PoolStatus::kOk && syncs == 0);          // fresh memory
  CHECK(pool.free(a, false) == PoolStatus::kOk && pool.settle(a) == PoolStatus::kForeign);
  CHECK(pool.malloc(&b, kUnit) && b == a && syncs == 0);                                     // reused at once
  CHECK(pool.settle(b) == PoolStatus::kOk && syncs == 1);
  CHECK(pool.settle(b) == PoolStatus::kOk && syncs == 1);                                    // nothing queued since
  CHECK(pool.free(b, false) == PoolStatus::kOk && pool.synchronize() && syncs == 2);
  CHECK(pool.malloc(&a, kUnit) && a == b && pool.settle(a) == PoolStatus::kOk && syncs == 2); // dropped before the wait
  CHECK(pool.free(a, true) == PoolStatus::kOk && pool.malloc(&c, kUnit) && c != a && pool.synchronize());
  CHECK(pool.malloc(&b, kUnit) && b == a && pool.settle(b) == PoolStatus::kOk && syncs == 3); // shared: settled by that
  std::printf("ok\n");
}
""")
    assert out == "ok\n"


def test_every_device_allocation_can_take_the_pools_blocks():
    """hipMalloc and hipMallocAsync are called in one place, behind the retry."""
    for f in sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.hip")):
        for i, line in enumerate(f.read_text().splitlines(), 1):
            code = line.split("//")[0]
            if "hipMalloc(" in code or "hipMallocAsync(" in code:
                assert f.name == "runtime.hip" and "pool_alloc_of(hipMalloc" in code, (f.name, i, line)


def test_padding_copies_stay_inside_a_grid(tmp_path):
    """The launch that pads a product's operands: under 2^26 blocks of 64 threads along x for any three matrices (HIP takes
    fewer than 2^32 threads there; 65535 products of 4096 x 17 x 17 would be 67 million blocks with one for every four
    rows), every row and product reached, and one block for each four rows where there is room."""
    cases = [(4096, 24, 8, 65535), (24, 24, 8, 65535), (65536, 24, 8, 4096), (16384, 24, 8, 16384), (131, 784, 8, 1), (1, 16, 8, 1),
             (2 ** 31 - 1, 2 ** 21, 8, 2 ** 31 - 1), (1, 2 ** 33, 16, 1), (5, 2 ** 31, 16, 3), (2048, 520, 8, 2 ** 26 + 1)]
    out = _run(tmp_path, r"""
#include "pad_blocks.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4) {
    const tsr950::PadBlocks b = tsr950::pad_blocks(atol(argv[i]), atol(argv[i + 1]), atoi(argv[i + 2]), atol(argv[i + 3]));
    std::printf("%u %u %u\n", b.bx, b.by, b.bz);
  }
}
""", *[x for c in cases for x in c])
    blocks = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(blocks) == len(cases)
    for (rows, ld, vec, batch), (bx, by, bz) in zip(cases, blocks):
        assert 3 * bx * by * bz < 2 ** 26
        assert bx * 64 * vec >= ld and 1 <= by <= -(-rows // 4) and 1 <= bz <= batch      # (rows and products in strides)
        if bx * -(-rows // 4) * batch <= 2 ** 24 and rows <= 65536:
            assert by == -(-rows // 4) and bz == batch
