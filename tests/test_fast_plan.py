"""The chunk rule of the specialised FP64 kernel (mcintegratorplusplus_amd/csrc/mci_fast_plan.hpp),
checked on the host for runs far longer than a GPU test could take: blocks (a Simple
accumulator's block is the whole run) of more than 2^31 steps must still be flushed exactly once
per block end, with every inner loop at most 2^30 steps."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mcintegratorplusplus_amd", "csrc")

PROG = r"""
#include "mci_fast_plan.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char **argv)
{
    const int64_t nsteps = std::atoll(argv[1]), B = std::atoll(argv[2]);
    const bool acc = std::atoi(argv[3]) != 0;
    int64_t s = 0, inblk = 0, flushes = 0, chunks = 0, maxlen = 0, minlen = INT64_MAX;
    while (s < nsteps) {
        const int len = mcid::fast_chunk_len(nsteps, s, B, inblk, acc);
        if (len < 1) { std::printf("bad %d\n", len); return 1; }
        maxlen = len > maxlen ? len : maxlen;
        minlen = len < minlen ? len : minlen;
        s += len;
        inblk += len;
        ++chunks;
        if (acc && inblk > B) { std::printf("crossed\n"); return 1; }
        if (acc && inblk == B) { ++flushes; inblk = 0; }
    }
    std::printf("%lld %lld %lld %lld %lld\n", (long long)s, (long long)flushes, (long long)chunks, (long long)maxlen, (long long)minlen);
    return 0;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src = d / "plan.cpp"
    src.write_text(PROG)
    exe = d / "plan"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)

    def run(nsteps, B, acc):
        out = subprocess.run([str(exe), str(nsteps), str(B), str(int(acc))], capture_output=True, text=True, check=True)
        return [int(v) for v in out.stdout.split()]
    return run


@pytest.mark.parametrize("nsteps,B,acc", [
    (10240, 160, True),              # the benchmark's blocks
    (2 ** 31 + 7, 2 ** 31 + 7, True),  # Simple accumulator beyond 2^31 (wrapped negative as an int)
    (2 ** 32 + 3, 2 ** 32 + 3, True),  # Simple accumulator beyond 2^32 (wrapped to 3 as an int)
    (3 * (2 ** 31 - 1), 2 ** 31 - 1, True),  # the largest Block size, three blocks
    (5, 5, True),
    (2 ** 33 + 1, 1, False),         # no accumulation (decorrelation)
])
def test_chunks_stay_32bit_and_flush_at_block_ends(plan, nsteps, B, acc):
    s, flushes, chunks, maxlen, minlen = plan(nsteps, B, acc)
    assert s == nsteps
    assert 1 <= minlen and maxlen <= 2 ** 30
    if acc:
        assert flushes == nsteps // B
    assert chunks >= -(-nsteps // 2 ** 30)


BITS = r"""
#include "mci_fast_plan.hpp"
#include <cstdio>
int main()
{
    for (long long n = 0; n <= 5000; ++n)
        std::printf("%lld %d %d %d %d\n", n, mcid::shared_index_bits(true, true, false, n), mcid::shared_index_bits(false, true, false, n),
                    mcid::shared_index_bits(true, false, false, n), mcid::shared_index_bits(true, true, true, n));
    return 0;
}
"""


def test_shared_index_bits_match_the_oracle(tmp_path):
    """The index bits the library takes from a native step's shared word (mci_fast_plan.hpp) and the
    oracle's rule (orc_shared_index_bits) agree: m for 2^m vectors up to 2^11, else -1 (Lemire);
    only native streams, vector moves, outside a MultiStepMove."""
    import ctypes as C

    from mcitest import Chain
    src = tmp_path / "bits.cpp"
    src.write_text(BITS)
    exe = tmp_path / "bits"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    rows = [list(map(int, ln.split())) for ln in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split("\n") if ln]
    for n, m, mt, allmove, ms in rows:
        exp = -1
        if n >= 1 and n & (n - 1) == 0 and n.bit_length() - 1 <= 11:
            exp = n.bit_length() - 1
        assert (m, mt, allmove, ms) == (exp, -1, -1, -1), n
    # the oracle, through contexts of 2^k coordinates with single-coordinate moves
    from mcitest import RNG_PHILOX, load
    lib = load("orc")
    lib.orc_shared_index_bits.argtypes = [C.c_void_p]
    for d in (1, 2, 3, 16, 24, 2048, 4096):
        c = Chain("orc", d, 1)
        c.setRng(RNG_PHILOX)
        c.setTrialMove(0, 1, 1, None)
        assert lib.orc_shared_index_bits(c.ctx) == rows[d][1], d
        c.setTrialMoveMultistep(2, 0, 1, 1, None)
        assert lib.orc_shared_index_bits(c.ctx) == -1


PARTS = r"""
#include "mci_fast_plan.hpp"
#include <cstdio>
#include <cstdlib>
#include <vector>
// a run of n steps on a buffer whose rows hold the running number of the output they were given
template <int LEFT> const char *run(int64_t n, int per)
{
    std::vector<int64_t> row(LEFT + mcid::MT_CH, -1);
    int64_t made = 0, taken = 0;
    const char *bad = nullptr;
    auto in = [&](int r) { if (r < 0 || r >= (int)row.size()) { bad = "row out of range"; } return bad == nullptr; };
    const mcid::MtEnd end = mcid::mt_parts<LEFT>(
        n, per,
        [&](int from, int to, int k) {
            if (k > LEFT) { bad = "more left over than the rows before a part"; return; }
            for (int r = 0; r < k; ++r) {
                if (in(from + r) && in(to + r)) { row[to + r] = row[from + r]; }
            }
        },
        [&](int q) {
            if (q != (made / mcid::MT_CH) % mcid::MT_SEG) { bad = "part out of order"; }
            for (int j = 0; j < mcid::MT_CH; ++j) { row[LEFT + j] = made++; }
        },
        [&](int r) {
            for (int j = 0; j < per; ++j) {
                if (in(r + j) && row[r + j] != taken + j) { bad = "not the next output"; }
            }
            taken += per;
        });
    if (taken != n * per) { return "steps"; }
    if (end.over != made - taken || end.over < 0 || end.over >= per + mcid::MT_CH) { return "outputs left over"; }
    if (n > 0 && end.next != (made - 1) % 312 + 1) { return "next element"; }
    return bad ? bad : "ok";
}
int main(int argc, char **argv)
{
    if (argc > 1) { // a long run: only the count of its steps and the parts' order
        int64_t steps = 0, parts = 0, wrong = 0;
        const mcid::MtEnd end = mcid::mt_parts<4>(std::atoll(argv[1]), 3, [](int, int, int) {},
                                                  [&](int q) { wrong += q != parts++ % mcid::MT_SEG; }, [&](int) { ++steps; });
        std::printf("%lld %lld %lld %d\n", (long long)steps, (long long)parts, (long long)wrong, end.over);
        return 0;
    }
#define SHAPE(S) for (int d = 1; d <= 4 * S; ++d) { for (int64_t n : N) { report(run<4 * S>(n, d + 1), d + 1, n); } }
    std::vector<int64_t> N;
    for (int64_t n = 0; n <= 700; ++n) { N.push_back(n); }
    N.push_back(20011);
    int fails = 0;
    auto report = [&](const char *r, int per, int64_t n) {
        if (r[0] != 'o' || r[1] != 'k') { if (fails++ < 10) { std::printf("%d outputs a step, %lld steps: %s\n", per, (long long)n, r); } }
    };
    SHAPE(1) SHAPE(2) SHAPE(3) SHAPE(4) SHAPE(6) SHAPE(8) SHAPE(12) SHAPE(16)
    for (int64_t n : N) { report(run<4>(n, 3), 3, n); }
    std::printf("%d failures\n", fails);
    return 0;
}
"""


@pytest.fixture(scope="module")
def parts(tmp_path_factory):
    d = tmp_path_factory.mktemp("parts")
    (d / "parts.cpp").write_text(PARTS)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(d / "parts.cpp"), "-o", str(d / "parts")], check=True)
    return lambda *a: subprocess.run([str(d / "parts"), *map(str, a)], capture_output=True, text=True, check=True).stdout


def test_generator_parts_follow_each_other_in_order(parts):
    """The lane-group kernels' order of making and taking a reference-stream generator's outputs
    (mt_parts): for every number of outputs a step takes in every form, and runs that end at every place
    of a part and of several rounds, each step takes the next outputs, parts are made in their order,
    every row lies in the buffer, and the end says which outputs were made and not taken."""
    assert parts() == "0 failures\n"


def test_generator_parts_in_a_run_past_32_bits(parts):
    """... and a run of more than 2^32 steps is one run: it neither stops short nor starts a part anew."""
    n = 2 ** 32 + 3
    made = -(-3 * n // 52)
    assert parts(n) == f"{n} {made} 0 {52 * made - 3 * n}\n"
