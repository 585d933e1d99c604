"""The host-side plan of an attention call (attn_plan in csrc/attention.hip), through the library without a GPU: the
scratch it asks for covers its records, is the same at every position of a cache (a prompt's later chunk, or a graph
captured after an early call, must not outgrow it), and calls take the kernel that measured faster."""
import collections
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "attention.hpp"
int main() {
  xtg::hip::DevKv c;
  int n_q, heads, window, fixed, ring, fp8;
  long long pos0;
  while (std::scanf("%d %d %lld %d %d %d %d %lld %d %d", &c.kv_heads, &c.head_dim, &c.slots, &ring, &fp8, &n_q, &heads,
                    &pos0, &window, &fixed) == 10) {
    c.ring = ring, c.fp8 = fp8, c.slots_pad = int((c.slots + 31) / 32 * 32);
    const xtg::hip::AttnPlan p = xtg::hip::attn_plan(c, n_q, heads, pos0, window, fixed != 0);
    std::printf("%d %d %d %d %d %d %zu %zu\n", p.tiles, p.splits, int(p.quads), int(p.few), p.own, p.run, p.used_floats(),
                p.part_floats());
  }
}
"""
Plan = collections.namedtuple("Plan", "tiles splits shared few own run used floats")


@pytest.fixture(scope="module")
def plans(pkg, tmp_path_factory):
    """plans([(kv_heads, head_dim, slots, ring, fp8, n_q, heads, pos0, window, fixed)]) -> [Plan]"""
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "xtier-go_amd", "csrc"), str(d / "plan.cpp"), pkg.LIB_PATH,
                    "-Wl,-rpath," + os.path.dirname(pkg.LIB_PATH), "-L/opt/rocm/lib", "-lamdhip64", "-o",
                    str(d / "plan")], check=True)

    def run(calls):
        text = "\n".join(" ".join(str(int(v)) for v in c) for c in calls) + "\n"
        env = {k: v for k, v in os.environ.items() if not k.startswith("XTG_")}
        r = subprocess.run([str(d / "plan")], input=text, capture_output=True, text=True, check=True, env=env)
        out = [Plan(*map(int, line.split())) for line in r.stdout.splitlines()]
        assert len(out) == len(calls)
        return out

    return run


@pytest.mark.parametrize("heads,kv,d", [(32, 8, 128), (16, 4, 256), (16, 8, 64), (8, 8, 128), (2, 1, 128), (64, 8, 256)])
@pytest.mark.parametrize("slots,ring,window", [(1040, 1, 1024), (1088, 1, 1024), (700, 1, 0), (9000, 0, 0), (9000, 0, 1024)])
def test_scratch_is_the_same_at_every_position(plans, heads, kv, d, slots, ring, window):
    for n_q in (1, 8, 20, 48, 130, 188, 512):
        last = 3 * slots if ring else slots - n_q
        if last < 0:
            continue
        at = sorted({0, 1, 31, 33, 512, 1000, 1023, 1024, 1025, slots // 2, slots - 1, slots, slots + 1, last} & set(range(last + 1)))
        for fp8 in (0, 1):
            ps = plans([(kv, d, slots, ring, fp8, n_q, heads, pos, window, 0) for pos in at])
            assert len({p.floats for p in ps}) == 1, (n_q, list(zip(at, ps)))
            assert all(p.used <= p.floats and p.splits <= p.tiles for p in ps)


def test_the_allocation_free_call_needs_what_it_writes(plans):
    """One own-key record per 128 keys and the splits of a full cache, whichever kernel takes the own keys: 48 rows of 256
    heads of 128 over 32 KV heads fit the 16 MiB array with one split."""
    calls = [(32, 128, 4096, 0, 0, 48, 256, 2000, 0, 1)]
    calls += [(kv, d, 1040, 1, 0, n, kv * group, 3000, 1024, 1) for d in (64, 128, 256) for kv, group in ((8, 4), (2, 8), (4, 1))
              for n in (1, 8, 9, 33, 48, 49, 100, 128, 129, 250)]
    for call, p in zip(calls, plans(calls)):
        assert p.used == p.floats and p.own == -(-call[5] // 128), (call, p)
    assert plans(calls[:1])[0].floats * 4 == 32 * 12 * 2 * 32 * 130 * 4 < 16 << 20


@pytest.mark.parametrize("heads,kv,d,last", [
    (16, 8, 64, 48), (8, 1, 64, 48), (32, 32, 64, 48), (8, 8, 128, 48), (2, 1, 128, 52), (32, 8, 128, 52), (64, 8, 128, 52),
    (4, 4, 256, 20), (8, 4, 256, 28), (16, 4, 256, 36), (8, 1, 256, 33)])
def test_calls_of_few_rows_keep_the_few_row_kernel(plans, heads, kv, d, last):
    """Up to the last rows at which it measured no slower than the tiled kernel."""
    for window in (0, 1024):
        ps = plans([(kv, d, 1040, 1, 0, n, heads, 500, window, 0) for n in (9, last, last + 1)])
        assert [p.few for p in ps] == [1, 1, 0] and ps[0].own == ps[1].own == 1


@pytest.mark.parametrize("heads,kv,d,slots,ring,ctx,n,shared", [
    (32, 8, 128, 2100, 0, 1500, 256, 0), (32, 8, 128, 2100, 0, 1500, 320, 1), (32, 8, 128, 6600, 0, 6000, 128, 1),
    (32, 8, 128, 1088, 1, 5000, 256, 0), (16, 4, 256, 1040, 1, 5000, 128, 0), (16, 4, 256, 1040, 1, 5000, 256, 1),
    (2, 1, 128, 6600, 0, 6000, 384, 0), (8, 8, 128, 2100, 0, 1500, 320, 0), (8, 8, 128, 6600, 0, 6000, 512, 1),
    (16, 8, 64, 2100, 0, 1500, 192, 0), (64, 8, 256, 2100, 0, 1500, 160, 1), (8, 1, 64, 2100, 0, 1500, 256, 0),
    (32, 8, 128, 6600, 0, 6000, 120, 0)])
def test_tiles_are_shared_where_that_measured_faster(plans, heads, kv, d, slots, ring, ctx, n, shared):
    """Calls whose two scans measured at least 8 % apart (the last is below the rows that share), and the most splits a
    work-group per CU allows."""
    p = plans([(kv, d, slots, ring, 0, n, heads, ctx, 1024 if ring else 0, 0)])[0]
    assert p.shared == shared
    if shared:
        blocks = -(-n // (32 // (heads // kv)))
        assert p.splits <= max(1, 256 // (kv * -(-blocks // 4)))


@pytest.mark.parametrize("heads,kv,d,n,run", [(32, 8, 128, 224, 64), (32, 8, 128, 512, 96), (16, 4, 256, 188, 32),
                                              (16, 4, 256, 512, 128), (64, 8, 128, 300, 64), (128, 16, 128, 100, 64)])
def test_runs_of_own_keys_are_the_ones_that_measured_fastest(plans, heads, kv, d, n, run):
    """Calls whose fastest run measured at least 4 % faster than the next (a run either way)."""
    assert plans([(kv, d, 4096, 0, 0, n, heads, 0, 0, 0)])[0].run == run
