"""Which slab and block a workgroup takes (fused_place_even,
fused_place_falling) and which grids take which: on the CPU, that every block is
taken once, how evenly the XCDs are loaded, and the edges of the rules; on the
GPU, the outputs of causal grids whose slabs are dealt over the XCDs."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "cuda_fused_attention_amd", "csrc")

# stdout: bad placements, then the largest share of an XCD over the average, of
# the falling order and of the even one, in the work of causal blocks (block b of
# n takes n - b) and in blocks, then the most slabs that an XCD reads of those
# left over where they are dealt by block number.
PROGRAM = r'''
#include "fa_fused_schedule.hpp"
#include <algorithm>
#include <cstdio>
#include <set>
#include <vector>
using namespace fa;
int main() {
    long bad = 0;
    double worst[2] = {0, 0}, count[2] = {0, 0};
    size_t most = 0;
    for (int slabs = 1; slabs <= 70; ++slabs)
        for (int n = 1; n <= 300; ++n)
            for (int falling = 0; falling < 2; ++falling) {
                std::vector<int> seen(slabs * n);
                double work[kXcds] = {}, blocks[kXcds] = {}, total = 0;
                std::set<int> left[kXcds];
                for (int x = 0; x < slabs * n; ++x) {
                    const FusedPlace p = falling ? fused_place_falling(x, slabs, n) : fused_place_even(x, slabs, n);
                    if (p.slab < 0 || p.slab >= slabs || p.block < 0 || p.block >= n || seen[p.slab * n + p.block]++) {
                        ++bad;
                        continue;
                    }
                    work[x % kXcds] += n - p.block;
                    blocks[x % kXcds] += 1;
                    total += n - p.block;
                    if (p.slab >= slabs / kXcds * kXcds && p.block < n / kXcds * kXcds) left[x % kXcds].insert(p.slab);
                }
                if (slabs * n <= 256) continue;
                for (int c = 0; c < kXcds; ++c) {
                    worst[falling] = std::max(worst[falling], work[c] * kXcds / total);
                    count[falling] = std::max(count[falling], blocks[c] - slabs * n / kXcds);
                    if (falling && n >= 64) most = std::max(most, left[c].size());
                }
            }
    std::printf("%ld %.3f %.3f %g %g %zu\n", bad, worst[1], worst[0], count[1], count[0], most);
}
'''


def test_every_block_once_and_even_loads(tmp_path):
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    bad, falling, even, falling_blocks, even_blocks, slabs = subprocess.run(
        [str(exe)], capture_output=True, text=True, check=True).stdout.split()
    assert bad == "0"
    assert float(falling) <= 1.04 and float(even) > 1.8  # contiguous ranges of one slab: 15/8
    assert float(falling_blocks) <= 1 and float(even_blocks) <= 1
    assert int(slabs) <= 2


RULES = r'''
#include "fa_fused_schedule.hpp"
#include <cstdio>
using namespace fa;
int main() {
    const struct { int slabs, workgroups, seq_len; bool causal; int order; bool two; } want[] = {
        {8, 256, 2048, true, kFusedEven, false},    {8, 264, 2112, true, kFusedFalling, false},
        {8, 512, 4096, true, kFusedFalling, false}, {16, 512, 2048, true, kFusedFalling, false},
        {18, 504, 1792, true, kFusedFalling, true},
        {19, 513, 1728, true, kFusedFalling, true}, {19, 494, 1664, true, kFusedEven, true},
        {8, 576, 4608, true, kFusedFalling, false}, {8, 584, 4672, true, kFusedFalling, true},
        {9, 513, 3648, true, kFusedFalling, true},  {300, 300, 64, true, kFusedEven, true},
        {37, 259, 398, true, kFusedFalling, true},  {281, 281, 64, true, kFusedFalling, true},
        {282, 282, 64, true, kFusedEven, true},     {1, 251, 16064, true, kFusedFalling, false},
        {2, 246, 7872, true, kFusedFalling, false}, {3, 255, 5440, true, kFusedEven, false},
        {1, 251, 16064, false, kFusedEven, false},
        {8, 256, 2048, false, kFusedEven, false},   {8, 264, 2112, false, kFusedEven, true},
        {8, 544, 4352, false, kFusedEven, true},    {8, 552, 4416, false, kFusedEven, false},
        {8, 768, 6144, false, kFusedEven, false},   {8, 776, 6208, false, kFusedEven, true},
        {38, 760, 1279, false, kFusedEven, true},   {38, 760, 1280, false, kFusedEven, false}};
    int bad = 0;
    for (const auto& w : want)
        bad += fused_order(w.slabs, w.workgroups, 256, w.causal) != w.order ||
               fused_two_stages(w.slabs, w.workgroups, 256, w.seq_len, w.causal) != w.two;
    std::printf("%d", bad);
}
'''


def test_rules_at_their_edges(tmp_path):
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text(RULES)
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout == "0"


@pytest.mark.gpu
@pytest.mark.parametrize("H,N", [(1, 8200), (2, 7000)])
def test_one_round_of_dealt_slabs(fa_lib, oracle_mod, H, N):
    """Four KV groups, fewer workgroups than CUs."""
    from gpu_common import HOST_THREADS, from_dev, nan_like, say, to_dev

    say("one round of dealt slabs", H, N)
    q, k, v = oracle_mod.make_inputs(1, H, N, 64)
    dev = [to_dev(x) for x in (q, k, v)]
    o = nan_like(dev[0])
    assert fa_lib.launch_attention_fused_groups(*dev, o, (1, H, N, 64), True, 64, 4)
    acc = oracle_mod.compare(from_dev(o), oracle_mod.attention(q, k, v, True, threads=HOST_THREADS))
    assert acc.passed, (H, N, acc)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,N", [(3, 5500), (37, 398), (11, 1500), (1, 16450), (5, 7500)])
def test_causal_grids_of_dealt_slabs(fa_lib, oracle_mod, H, N, D):
    """64 rows: few slabs of many blocks (with a partial level of 6, 2 and 1), and
    more than 8 of few, one of them little more than a round; 37 and 5 slabs with two
    LDS stages at head_dim 128."""
    from gpu_common import HOST_THREADS, from_dev, nan_like, say, to_dev

    cus = fa_lib.query_tensorcore_v3(D)["compute_units"]
    assert cus < H * ((N + 63) // 64)
    say("dealt slabs", H, N, D)
    q, k, v = oracle_mod.make_inputs(1, H, N, D)
    dev = [to_dev(x) for x in (q, k, v)]
    o = nan_like(dev[0])
    assert fa_lib.launch_attention_fused(*dev, o, (1, H, N, D), True, rows_per_block=64)
    acc = oracle_mod.compare(from_dev(o), oracle_mod.attention(q, k, v, True, threads=HOST_THREADS))
    assert acc.passed, (H, N, D, acc)
