"""The 64-row kernel with two LDS stages per tensor (head_dim 128, more
workgroups than CUs): its stage schedule on the CPU, and its outputs against the
FP64 oracle and against the three-stage kernel, whose arithmetic it shares."""
import os
import subprocess

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "cuda_fused_attention_amd", "csrc")

# One group's walk: K_{jj+3} and V_{jj+2} are copied in block B of step jj,
# nothing is in flight at a step's barrier, K_2 is copied after the prologue's
# second barrier, and a base move reads no stage.
PROGRAM = r'''
#include "fa_fused_schedule.hpp"
#include <cstdio>
#include <vector>
using namespace fa;
constexpr int S = 2;
struct Stage { int tile = -1; bool landed = false; int landed_epoch = -1; };
long bad = 0;
int epoch = 0;
std::vector<Stage> ks, vs;
void dma(std::vector<Stage>& arr, int st, int tile, int consumed) {
    if (arr[st].tile >= 0 && arr[st].tile > consumed) ++bad;
    arr[st] = Stage{tile, false, -1};
}
void wait_all() {
    for (auto* a : {&ks, &vs})
        for (auto& s : *a)
            if (s.tile >= 0 && !s.landed) { s.landed = true; s.landed_epoch = epoch; }
}
void read(std::vector<Stage>& arr, int st, int tile) {
    if (arr[st].tile != tile || !arr[st].landed || arr[st].landed_epoch >= epoch) ++bad;
}
int main() {
    for (int cnt = 0; cnt <= 400; ++cnt) {
        ks.assign(S, Stage{}); vs.assign(S, Stage{}); epoch = 0;
        for (int x = 0; x < S; ++x) dma(ks, x, x, -1);
        for (int x = 0; x < kFusedVAhead; ++x) dma(vs, x % S, x, -1);
        wait_all(); ++epoch;
        if (cnt > 0) read(ks, 0, 0);
        wait_all(); ++epoch;
        int k_consumed = 0, k_pending = 1, v_consumed = -1, v_pending = -1;
        read(ks, 1, 1);
        dma(ks, 0, 2, k_consumed);
        fused_group_walk(cnt, [&](auto par, int jj) {
            if (decltype(par)::value % S != jj % S) ++bad;
            read(vs, jj % S, jj);
            v_pending = jj;
            WAIT(); ++epoch;
            v_consumed = v_pending; k_consumed = k_pending;
            dma(ks, (jj + kFusedKAhead) % S, jj + kFusedKAhead, k_consumed);
            dma(vs, (jj + kFusedVAhead) % S, jj + kFusedVAhead, v_consumed);
            read(ks, (jj + 2) % S, jj + 2);
            k_pending = jj + 2;
        });
    }
    std::printf("%ld\n", bad);
    return bad != 0;
}
'''


def replay(tmp_path, program, tag):
    src, exe = tmp_path / f"{tag}.cpp", tmp_path / tag
    src.write_text(program)
    r = subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return subprocess.run([str(exe)], capture_output=True, text=True)


def test_schedule(tmp_path):
    out = replay(tmp_path, PROGRAM.replace("WAIT()", "wait_all()"), "ok")
    assert out.returncode == 0 and out.stdout.strip() == "0", out.stdout
    # planted: a step that does not wait, copies one tile further ahead
    for tag, (old, new) in {"nowait": ("WAIT()", "(void)0"),
                            "ahead": ("dma(ks, (jj + kFusedKAhead) % S, jj + kFusedKAhead, k_consumed);",
                                      "dma(ks, (jj + kFusedKAhead + 1) % S, jj + kFusedKAhead + 1, k_consumed);")}.items():
        out = replay(tmp_path, PROGRAM.replace(old, new).replace("WAIT()", "wait_all()"), tag)
        assert out.returncode != 0 and out.stdout.strip() != "0", tag


@pytest.mark.gpu
@pytest.mark.parametrize("N", [1, 33, 64, 65, 130, 257])
@pytest.mark.parametrize("family", ["uniform", "stress", "scaled"])
def test_two_stage_outputs(fa_lib, oracle_mod, N, family):
    """More 64-row workgroups than CUs: every slab passes the oracle gate, and
    the first slabs equal, bit for bit, what the three-stage kernel gives for
    them alone (fewer workgroups than CUs). The stress and scaled families move
    the exponent base, which takes V from global memory here. Dense only for the
    bits at one round: causal grids of one round pair their rows, so there the
    keys are split at other tiles."""
    from gpu_common import HOST_THREADS, from_dev, nan_like, say, to_dev

    D, H = 128, 300
    cus = fa_lib.query_tensorcore_v3(128)["compute_units"]
    assert H > cus
    q, k, v = oracle_mod.make_inputs(1, H, N, D, family)
    for causal in (False, True):
        say("two stages", N, family, causal)
        ref = oracle_mod.attention(q, k, v, causal, threads=HOST_THREADS)
        dev = [to_dev(x) for x in (q, k, v)]
        o = nan_like(dev[0])
        assert fa_lib.launch_attention_fused(*dev, o, (1, H, N, D), causal, rows_per_block=64)
        got = from_dev(o)
        acc = oracle_mod.compare(got, ref)
        assert acc.passed, (N, family, causal, acc)
        if not causal:
            few = 20
            part = nan_like(dev[0][:, :few])
            assert fa_lib.launch_attention_fused(*(x[:, :few].contiguous() for x in dev), part, (1, few, N, D), causal,
                                                 rows_per_block=64)
            assert np.array_equal(from_dev(part), got[:, :few])


@pytest.mark.gpu
@pytest.mark.parametrize("N", [901, 1050])
@pytest.mark.parametrize("family", ["uniform", "stress", "scaled"])
def test_two_stage_long_walks(fa_lib, oracle_mod, N, family):
    """15 and 17 steps per group: more than one unrolled pass, with every step of
    it as the last of a causal block; the stress family moves the base far into a
    walk. Checked as in test_two_stage_outputs."""
    from gpu_common import HOST_THREADS, from_dev, nan_like, say, to_dev

    D, H, few = 128, 20, 5
    cus = fa_lib.query_tensorcore_v3(128)["compute_units"]
    assert few * ((N + 63) // 64) < cus < H * ((N + 63) // 64)
    q, k, v = oracle_mod.make_inputs(1, H, N, D, family)
    dev = [to_dev(x) for x in (q, k, v)]
    for causal in (False, True):
        say("two stages, long", N, family, causal)
        o = nan_like(dev[0])
        assert fa_lib.launch_attention_fused(*dev, o, (1, H, N, D), causal, rows_per_block=64)
        got = from_dev(o)
        acc = oracle_mod.compare(got, oracle_mod.attention(q, k, v, causal, threads=HOST_THREADS))
        assert acc.passed, (N, family, causal, acc)
        if not causal:
            part = nan_like(dev[0][:, :few])
            assert fa_lib.launch_attention_fused(*(x[:, :few].contiguous() for x in dev), part, (1, few, N, D), causal,
                                                 rows_per_block=64)
            assert np.array_equal(from_dev(part), got[:, :few])


@pytest.mark.gpu
def test_query_reports_the_two_stage_kernel(fa_lib):
    """Where v3 runs it: no spills, two workgroups per CU."""
    for causal in (False, True):
        seen = 0
        for shape in [(1, bh, 1100, 128) for bh in range(20, 60)] + [(1, 22, 1435, 128), (1, 20, 1557, 128)]:
            if fa_lib.tensorcore_v3_config(shape, causal) == (64, 2):
                info = fa_lib.query_tensorcore_v3_shape(shape, causal)
                assert info["local_bytes_per_thread"] == 0 and info["max_blocks_per_sm"] == 2, info
                assert info["shared_bytes_per_block"] == 80 * 1024 and info["agprs_per_thread"] >= 0
                seen += 1
        assert seen > 0, causal
