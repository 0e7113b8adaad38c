"""The host side of prompt attention (csrc/attention_prompt_plan.hpp), compiled
on its own: how the calls that its rule takes are cut into workgroups."""
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "barq-inference_amd", "csrc")
CUS = 256

MAIN = r"""
#include "attention_prompt_plan.hpp"
#include <algorithm>
#include <chrono>
#include <cstdio>
using namespace barq;
// shapes on stdin -> taken, ns of a plan (best of five), G, groups, tiles, chunk, stride, blocks of every tile
int main() {
    long long nh, nkv, hd, q, kv;
    while (scanf("%lld %lld %lld %lld %lld", &nh, &nkv, &hd, &q, &kv) == 5) {
        ApPlan p;
        long long ns = 1LL << 60;
        for (int i = 0; i < 5; i++) {
            const auto t0 = std::chrono::steady_clock::now();
            p = ap_plan(nh, nkv, hd, q, kv, 256, 0);
            ns = std::min(ns, (long long)std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now() - t0).count());
        }
        printf("%d %lld %d %d %d %d %d", (int)ap_path(nh, nkv, hd, q, kv, p), ns, p.G, p.groups, p.tiles, p.chunk, p.stride);
        for (int t = 0; t < p.tiles; t++) printf(" %d", ap_tile_blocks(t, p.G, q, kv, kv > q ? kv - q : 0));
        printf("\n");
    }
}
"""

HEADS = [(32, 8), (32, 4), (32, 32), (24, 8), (16, 8), (8, 1), (14, 2), (71, 1), (15, 5), (6, 4), (9, 3), (1, 1), (3, 1)]


def shapes():
    r = random.Random(3)
    out = [(14, 2, 64, 8, 4000), (71, 1, 64, 4, 4000), (15, 5, 64, 16, 4000), (32, 8, 128, 8, 4000), (8, 1, 128, 64, 131072),
           (32, 8, 128, 2048, 2048), (32, 8, 64, 200, 1000), (1, 1, 64, 2, 100000),
           (14, 2, 64, 8, 4008), (16, 8, 128, 59, 504), (32, 8, 128, 12, 4012), (32, 8, 128, 64, 564), (32, 8, 64, 24, 4024),
           (32, 32, 128, 6, 4006), (32, 32, 128, 2, 4002), (24, 8, 128, 7, 1289), (71, 1, 64, 4, 4004), (24, 8, 128, 67, 174),
           (14, 2, 128, 180, 180), (28, 4, 64, 151, 151), (32, 8, 128, 40, 40), (28, 4, 64, 5, 3798), (28, 4, 128, 8, 1657)]
    for _ in range(400):
        q = int(round(2 ** r.uniform(1, 11)))
        out.append((*r.choice(HEADS), r.choice([64, 128]), q, q + r.choice([0, int(round(2 ** r.uniform(4, 14)))])))
    return out


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, exe = d / "main.cpp", d / "plan"
    src.write_text(MAIN)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    text = "".join(" ".join(map(str, s)) + "\n" for s in shapes())
    lines = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    rows = [list(map(int, line.split())) for line in lines]
    return [(s, bool(r[0]), *r[1:7], r[7:]) for s, r in zip(shapes(), rows)]


def test_tiles_cover_the_rows(plans):
    for s, _, _, g, groups, tiles, chunk, stride, nbs in plans:
        nh, nkv, _, q, kv = s
        assert g * groups == nh and (nkv == groups or nh % nkv), s
        assert len(nbs) == tiles and (tiles - 1) * 128 < q * g <= tiles * 128, s
        assert max(nbs) == (kv + 31) // 32, s
        # the workspace holds every piece, wherever the rows start
        assert chunk == 0 and stride == 1 or chunk * stride >= (kv + 31) // 32 > chunk, s


def test_calls_that_the_rule_takes_fill_the_cus(plans):
    """No workgroup walks much more than a CU's share of the position blocks: at
    most twice that (two workgroups share a CU) and three blocks of fixed part."""
    taken = 0
    for s, take, _, _, groups, _, chunk, _, nbs in plans:
        if not take:
            continue
        taken += 1
        share = sum(nbs) * groups / CUS
        assert max(nbs) <= 2 * share + 3 or (0 < chunk <= 2 * share + 3), (s, chunk, max(nbs), share)
    assert taken > 100


def test_a_plan_takes_microseconds(plans):
    """A server's shapes change with every step, so a plan is part of the call:
    at most some 8 us on an idle core, half a microsecond for a few rows (a
    simulation of the launch took 0.4 to 8 ms).  Bars four times that and more,
    for a busy machine."""
    for s, _, ns, *_ in plans:
        assert ns < 40000, (s, ns)
    few = [ns for s, _, ns, *_ in plans if s[3] <= 16]
    assert sorted(few)[len(few) // 2] < 5000, sorted(few)


def test_the_rule_takes_the_faster_kernel(plans):
    """Calls measured on MI355X, us of the decode kernel and of the prompt one:
    the prompt one is not taken where it is over 15 % slower, and always where
    the other takes twice as long."""
    measured = {(14, 2, 64, 8, 4008): (16, 20), (16, 8, 128, 59, 504): (13, 22), (32, 8, 128, 12, 4012): (44, 33), (32, 8, 128, 64, 564): (23, 25),
                (32, 8, 64, 24, 4024): (40, 26), (32, 32, 128, 6, 4006): (70, 43), (32, 32, 128, 2, 4002): (33, 43),
                (24, 8, 128, 7, 1289): (31, 22), (71, 1, 64, 4, 4004): (55, 23), (24, 8, 128, 67, 174): (15, 19),
                (14, 2, 128, 180, 180): (17, 19), (28, 4, 64, 151, 151): (21, 14), (32, 8, 128, 40, 40): (8, 16), (32, 8, 128, 2048, 2048): (1261, 210),
                (28, 4, 64, 5, 3798): (37, 19), (28, 4, 128, 8, 1657): (32, 23)}
    takes = {s: take for s, take, *_ in plans}
    for s, (rows, prompt) in measured.items():
        assert not takes[s] or prompt <= 1.15 * rows, s
        assert takes[s] or rows < 2 * prompt, s
