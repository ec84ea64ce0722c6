# SPDX-License-Identifier: Apache-2.0
"""What the device entry points take of a workspace, from their own layout functions on a
machine without a GPU (tests/c/k3_ws_sizes.c, at the MI355X's 256 CUs)."""
import glob
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "kimi-k3-in-c_amd")
MIB = 1 << 20


@pytest.fixture(scope="module")
def sizes(tmp_path_factory):
    """[(least, takes, k3d_moe_ws, router least, takes, k3d_router_ws, most over 1..T, router most)]
    of (T, hidden, inter, experts, topk, prec)."""
    objs = [o for o in glob.glob(os.path.join(PKG, "_build", "*.o")) if not o.endswith("k3_devapi.o")]
    if not objs:
        subprocess.run(["make", "-j8", "-C", PKG], check=True)
        objs = [o for o in glob.glob(os.path.join(PKG, "_build", "*.o")) if not o.endswith("k3_devapi.o")]
    exe = str(tmp_path_factory.mktemp("ws") / "k3_ws_sizes")
    subprocess.run(["gcc", "-std=gnu99", "-O2", "-Wall", "-Wextra", "-Wno-unused-parameter", "-Werror",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(ROOT, "tests", "c", "k3_ws_sizes.c"), *objs, "-o", exe, "-Wl,--wrap=k3k_cu_count",
                    "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64", "-lstdc++", "-lgomp", "-lpthread", "-lm"],
                   check=True)

    def ask(shapes, step=1):
        text = "".join("%d %d %d %d %d %d\n" % s for s in shapes)
        out = subprocess.run([exe, "256", str(step)], input=text, capture_output=True, text=True, check=True).stdout
        rows = [tuple(map(int, ln.split())) for ln in out.splitlines()]
        assert len(rows) == len(shapes)
        return rows
    return ask


def al(n):
    return (n + 255) // 256 * 256


def plain_need(T, hidden, inter, n, k, prec, router):
    """One list of passes of at least 8 assignments, 16 where the widths are no multiples of 512, and
    the router's scratch."""
    N = T * k
    jobs = min(N, n)
    passes = jobs + N // (16 if hidden % 512 or inter % 512 else 8) + 1
    b = (2 if prec == 0 else 1) * (al(T * hidden * 2) + al(N * inter * 2)) + al((n + 1) * 4) + al(N * 4)
    b += 3 * al(jobs * 4) + 2 * al(passes * 4) + al(N * hidden * 4) + (al(N * 2 * inter * 4) if N <= 16 else 0)
    return b + router


# (token count, shape) around the largest batches of the static workspace that need no more than it holds
@pytest.mark.parametrize("shape", [(160, 7168, 2048, 384, 4, 0), (194, 7168, 1024, 384, 4, 0), (192, 3584, 3072, 896, 4, 0),
                                   (285, 4096, 3584, 512, 2, 1)])
def test_static_workspace_holds(sizes, shape):
    (least, takes, ws, *_), = sizes([shape])
    assert least <= 40 * MIB and least <= takes <= ws


def test_least_scratch(sizes):
    """A call is never refused for scratch that its fp64 router partials and one pass list would
    have left free, whatever partials and lists it would rather take."""
    rng = random.Random(7)
    shapes = [(rng.randint(1, 1023), 32 * rng.randint(1, 256), 32 * rng.randint(1, 128), rng.randint(1, 1024),
               rng.randint(1, 16), rng.randint(0, 1)) for _ in range(150)]
    shapes += [(rng.randint(1, 1023), 512 * rng.randint(1, 16), 512 * rng.randint(1, 8), rng.choice((60, 128, 384, 896)),
                rng.choice((2, 4, 8, 16)), rng.randint(0, 1)) for _ in range(150)]
    for s, (least, takes, ws, rleast, rtakes, rws, _, _) in zip(shapes, sizes(shapes)):
        N, n = s[0] * s[4], s[3]
        hist = al((N + 511) // 512 * n * 4) if N > 2048 and n <= 1024 else 0
        assert least <= takes <= ws and rleast <= rtakes <= rws, s
        assert least <= plain_need(*s, rleast) + al((4 + 4 * 8) * 4) + hist, s


def test_size_covers_smaller_batches(sizes):
    """k3d_moe_ws and k3d_router_ws of T tokens are enough for any batch of up to T, whichever
    partials and pass lists it takes."""
    rng = random.Random(11)
    shapes = [(127, 7168, 512, 384, 8, 0), (7, 7168, 512, 384, 8, 0), (255, 7168, 512, 128, 8, 0), (548, 7168, 512, 64, 8, 0)]
    shapes += [(rng.randint(1, 1500), 512 * rng.randint(1, 16), 512 * rng.randint(1, 8), rng.choice((3, 60, 64, 128, 384, 896, 1400)),
                rng.choice((1, 2, 4, 8, 16)), rng.randint(0, 1)) for _ in range(120)]
    shapes += [(rng.randint(1, 1500), 32 * rng.randint(1, 256), 32 * rng.randint(1, 128), rng.randint(1, 2048),
                rng.randint(1, 24), rng.randint(0, 1)) for _ in range(120)]
    for s, (_, _, ws, _, _, rws, most, rmost) in zip(shapes, sizes(shapes)):
        assert rmost <= rws and most <= ws, s
    # long prompts, past the last change of a chunk count (49,932 tokens: the int8 kernels' last)
    shapes = [(t, h, 512, n, 2, 1) for t in (20000, 60000) for h in (512, 7168) for n in (40, 64, 896)]
    for s, (_, _, ws, _, _, rws, most, rmost) in zip(shapes, sizes(shapes, 32)):
        assert rmost <= rws and most <= ws, s
