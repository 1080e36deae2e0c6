"""The attn_bias requests of hstu_bwd_kv_fused_kernel (hstu_bias_requests.h), compiled for the host and replayed: every byte that a lane's
requests fetch, the one behind the last step included, belongs to the plane of a query head of that wavefront, and a step's request
names the head and the rows of the step."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ops-rec_amd", "csrc")

# A raw buffer load fetches the 4-byte words that lie below the descriptor's size and returns 0 for the others.  The sequence has
# sq <= max_q rows and sk <= max_k keys; a causal mask starts the sweep at the first sub-tile that sees the tile, context rows put a gap
# in it.  Prints how many requests fetched something they should not have, and the first of them.
REPLAY = r"""
#include <cstdio>
#include "hstu_bias_requests.h"

int main()
{
    const uint64_t kBase = 1ull << 40;
    long bad = 0, fetched = 0;
    for (int ratio = 1; ratio <= 4; ratio *= 2) {
        for (int max_k = 2; max_k <= 512; max_k += 2) {
            const int max_q = max_k % 3 == 0 ? max_k : (max_k + 95) / 2;
            const int64_t size = static_cast<int64_t>(max_q) * max_k * 2;
            const int n_qsub = (max_q + 31) / 32;
            for (int c0 = 0; c0 < max_k; c0 += 128) {
                for (int sweep = 0; sweep < 3; ++sweep) {  // all sub-tiles, a causal sweep, one with context rows in front
                    const int causal = c0 / 32 < n_qsub ? c0 / 32 : n_qsub;
                    const int first = sweep == 1 ? causal : 0;
                    const bool gap = sweep == 2 && causal > 1;
                    const int steps = ratio * (n_qsub - first - (gap ? causal - 1 : 0));
                    if (steps == 0) {
                        continue;
                    }
                    for (int lane = 0; lane < 4 * 64; ++lane) {
                        const int cw0 = c0 + lane / 64 * 32, ln = lane % 32, lh = lane / 32 % 2;
                        hstu::BiasRequests r;
                        r.plane = kBase;
                        r.pitch = max_k * 2;
                        r.size = static_cast<uint32_t>(size);
                        r.x = r.first = first;
                        r.skip_from = gap ? 1 : -1;
                        r.skip_to = gap ? causal : -1;
                        r.end = n_qsub;
                        r.left = steps;
                        r.set_lane(max_k, cw0, ln, lh);
                        int x = first;
                        uint64_t plane = kBase;
                        for (int i = 0; i <= steps; ++i) {  // (one request per step, a step ahead, and none left behind the last)
                            bool wrong = i < steps && (r.x != x || r.plane != plane);
                            for (int piece = 0; piece < 64; piece += 4) {
                                if (piece >= 16 && (piece < 32 || piece >= 48)) {
                                    continue;
                                }
                                const uint32_t off = r.offset() + piece;
                                if (off >= r.bytes()) {
                                    continue;
                                }
                                ++fetched;
                                const int64_t at = static_cast<int64_t>(r.plane - kBase) + off;
                                wrong = wrong || i == steps || at < 0 || at + 4 > ratio * size || off / r.pitch < static_cast<uint32_t>(x * 32 + ln);
                            }
                            if (wrong && bad++ == 0) {
                                std::printf("ratio %d, max_seq_len_k %d, key %d, lane %d, request %d of %d: plane %lld, offset %u\n", ratio, max_k,
                                            cw0, lane % 64, i, steps, (long long)((r.plane - kBase) / size), r.offset());
                            }
                            r.advance();
                            if (++x == r.skip_from) {
                                x = r.skip_to;
                            }
                            if (x >= n_qsub) {
                                x = first;
                                plane += size;
                            }
                        }
                    }
                }
            }
        }
    }
    std::printf("%ld of %ld\n", bad, fetched);
    return bad != 0 || fetched == 0;
}
"""


def test_no_request_leaves_the_planes_of_its_heads(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++ on this host")
    source, program = tmp_path / "replay.cpp", tmp_path / "replay"
    source.write_text(REPLAY)
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(source), "-o", str(program)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout
