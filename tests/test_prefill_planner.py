"""The prefill planner's tail split (planner.cpp) on the CPU, compiled with the
host compiler: which blocks are split, against the rule written out in full
here (every candidate's whole schedule), and what looking for them costs."""
import heapq
import os
import random
import subprocess

import pytest

from dendrite_amd import build as dbuild

MAIN = r"""
#include <chrono>
#include <cstdio>
#include <numeric>
#include "planner.hpp"
int main() {   // d hq hkv causal chunk_pages repetitions batch kv_len... q_len... a line
    unsigned d, hq, hkv, causal, chunk, reps, B;
    while (scanf("%u%u%u%u%u%u%u", &d, &hq, &hkv, &causal, &chunk, &reps, &B) == 7) {
        std::vector<uint32_t> kv(B), q(B), ip(1, 0);
        for (auto* v : {&kv, &q})
            for (auto& x : *v)
                if (scanf("%u", &x) != 1) return 1;
        for (auto x : kv) ip.push_back(ip.back() + (x + 15) / 16);
        std::vector<uint32_t> ix(ip.back());
        std::iota(ix.begin(), ix.end(), 0u);
        dh::PrefillInput in;
        in.batch = B, in.indptr = ip.data(), in.indices = ix.data(), in.kv_len = kv.data(), in.q_len = q.data();
        in.num_pool_pages = ip.back(), in.hq = hq, in.hkv = hkv, in.causal = causal, in.chunk_pages = chunk;
        in.group_rows = dh::group_rows(false, int(d)), in.wg_slots = dh::prefill_slots(int(d));
        dh::HostPlan hp;
        std::string err;
        double best = 1e30;
        for (unsigned r = 0; r < reps; ++r) {
            const auto t0 = std::chrono::steady_clock::now();
            if (dh::build_prefill_plan(in, hp, err)) return 2;
            best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
        }
        printf("%zu %zu %u %.2f\n", hp.items.size(), hp.split_rows.size(), hp.num_slots, best);
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """plans(lines) -> (items, split rows, slots, us) of each plan."""
    tmp = tmp_path_factory.mktemp("planner")
    (tmp / "main.cpp").write_text(MAIN)
    exe = str(tmp / "plans")
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{os.path.join(dbuild.ROOT, 'include')}", f"-I{dbuild.CSRC}",
                    str(tmp / "main.cpp"), os.path.join(dbuild.CSRC, "planner.cpp"), "-o", exe], check=True)

    def run(lines):
        text = "".join(" ".join(map(str, ln)) + "\n" for ln in lines)
        # Memory freed stays with the process, so that no plan pays for fresh pages.
        env = dict(os.environ, MALLOC_MMAP_THRESHOLD_=str(1 << 30), MALLOC_TRIM_THRESHOLD_=str(1 << 30))
        out = subprocess.run([exe], input=text, text=True, capture_output=True, check=True, env=env).stdout.splitlines()
        assert len(out) == len(lines)
        return [tuple(float(x) if "." in x else int(x) for x in ln.split()) for ln in out]
    return run


def _makespan(cost, cols):
    free = [0] * cols
    for c in cost:
        heapq.heapreplace(free, free[0] + c)
    return max(free)


def expected(d, hq, hkv, causal, kv, q):
    """(items, split rows, slots) of a plan of whole blocks by the rule."""
    r, slots = hq // hkv, 256 if d == 256 else 512
    tpb = (64 if d == 256 else 128) // r
    blk = []                     # pages, last chunk start, tiles, queries
    for k, n in zip(kv, q):
        for i0 in range(0, n, tpb):
            i1 = min(n, i0 + tpb)
            first, last = (k - n + i0 + 1, k - n + i1) if causal else (k, k)
            blk.append(((last + 15) // 16, (first - 1) // 16, ((i1 - i0) * r + 15) // 16, i1 - i0))
    whole = (len(blk) * hkv, 0, sum(q))
    n, cols = len(blk), max(1, slots // hkv)
    rem = n % cols
    assert n * hkv >= 512
    if n // cols == 0 or n // cols >= 8 or rem == 0:
        return whole
    order = sorted(range(n), key=lambda i: -blk[i][0] * (2 + blk[i][2]))
    base = [blk[i][0] * (2 + blk[i][2]) + 80 for i in order]
    end = _makespan(base, cols)
    best, got = end - end // 20, whole
    if sum(base) // cols >= best:
        return whole
    for m in (rem, rem + cols // 4):
        for ch in (16, 32, 64, 128):
            if m >= n:
                continue
            cost, states, items, rows = base[:n - m], 0, n - m, 0
            for i in order[n - m:]:
                pages, plast, tiles, tokens = blk[i]
                k = plast // ch
                cost += [ch * (2 + tiles) + 240] * k + [(pages - k * ch) * (2 + tiles) + 80 + (160 if k else 0)]
                states += (k + 1) * tokens if k else 0
                rows += tokens if k else 0
                items += k + 1
            if 2 * states > sum(q):
                continue
            e = _makespan(sorted(cost, reverse=True), cols) + 120 + 8 * states * hkv // slots
            if e < best:
                best, got = e, (items * hkv, rows, states)
    return got


def _shapes():
    rng = random.Random(11)
    out = [(64, 64, 8, 1, [1500], [1066]), (64, 128, 8, 1, [1500], [536]), (128, 32, 8, 1, [30300], [2300]),
           (128, 32, 1, 1, [31000], [3000]), (128, 32, 8, 1, [4756, 5898, 5192], [529, 900, 670])]
    while len(out) < 60:
        d, hkv, r = rng.choice([64, 128, 256]), rng.choice([1, 2, 4, 8, 16, 32]), rng.choice([1, 4, 8, 16])
        tpb, cols = (64 if d == 256 else 128) // r, max(1, (256 if d == 256 else 512) // hkv)
        n, batch = cols * rng.randint(1, 3) + rng.randint(1, max(1, cols // 3)), rng.choice([1, 1, 3])
        q = [max(1, int(n * tpb / batch * rng.uniform(0.8, 1.2))) for _ in range(batch)]
        kv = [x + rng.choice([0, 2000, 9000]) for x in q]
        if n < 1200 and max(kv) <= 30000 and sum((x + tpb - 1) // tpb for x in q) * hkv >= 512:
            out.append((d, r * hkv, hkv, rng.choice([1, 1, 0]), kv, q))
    return out


def test_tail_split_follows_the_rule(plans):
    shapes = _shapes()
    got = plans([(d, hq, hkv, causal, 0, 1, len(q), *kv, *q) for d, hq, hkv, causal, kv, q in shapes])
    want = [expected(*s) for s in shapes]
    assert [g[:3] for g in got] == want
    assert sum(w[1] > 0 for w in want) >= 10 and sum(w[1] == 0 for w in want) >= 10


@pytest.mark.parametrize("shape", [(128, 32, 1, [31000], [3000]), (128, 32, 8, [30300], [2300]),
                                   (64, 32, 4, [600 + 70 * i for i in range(12)], [600 + 70 * i for i in range(12)])],
                         ids=["750-blocks", "72-blocks", "12-prompts"])
def test_planning_without_a_split_stays_cheap(plans, shape):
    """Plans that end up whole: looking for a tail split adds less than half
    to the planning time of the same items asked for by their chunk size
    (trying every candidate's schedule took 20 times as long)."""
    d, hq, hkv, kv, q = shape
    runs = [plans([(d, hq, hkv, 1, chunk, 40, len(q), *kv, *q) for chunk in (0, 2000)]) for _ in range(3)]
    assert all(a[0] == b[0] and a[1] == 0 for a, b in runs)
    assert min(a[3] for a, _ in runs) < 1.5 * min(b[3] for _, b in runs)
