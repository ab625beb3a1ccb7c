"""Host-side logic of the Python drop-ins that needs no GPU: configuration checks and
the refusals of configurations that have no HIP path, and what the compiler makes of the
inline LDS DMA."""

import re
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest


def test_output_role_repair_config():
    """repair_features="output_role" (reference n8_v6.py:1246-1290) is accepted with the Q role
    ranks the role-feature apply kernel takes (16, 32, 48, 64) and refused with others."""
    from sparsepr_amd.n8_v6 import N8V6Config

    N8V6Config(repair_features="output").validate()
    N8V6Config(repair_features="output_role").validate()
    N8V6Config(repair_features="output_role", role_q_rank=32).validate()
    with pytest.raises(NotImplementedError, match="role_q_rank"):
        N8V6Config(repair_features="output_role", role_q_rank=40).validate()
    with pytest.raises(ValueError, match="repair_features must be"):
        N8V6Config(repair_features="bogus").validate()


def test_route_feature_dims_the_kernels_take():
    """The role-space k-means runs on feature dims that are multiples of 16 up to 128: other
    Q role ranks or K (+ V) feature counts are refused before any launch, naming the limit."""
    from sparsepr_amd.n8_v6 import N8V6Config, N8V6Core

    N8V6Core(N8V6Config())._check_route_config(128)
    N8V6Core(N8V6Config(role_k_rank=32, role_v_rank=16, role_v_weight=0.5))._check_route_config(64)
    for cfg, dim in ((N8V6Config(role_q_rank=40), 128), (N8V6Config(role_k_rank=24), 128),
                     (N8V6Config(role_k_rank=64, role_v_rank=72, role_v_weight=0.5), 128),
                     (N8V6Config(), 96)):
        with pytest.raises(NotImplementedError, match="multiple of 16"):
            N8V6Core(cfg, validate=False)._check_route_config(dim)


# A descriptor put together by v_readlane right before the inline DMA, and the compiler's own DMA,
# with the same LDS base before and after it.
_DMA_PROBE = """
#include "spr_common.h"
__global__ void probe(const int32_t* words, const int32_t* src, int32_t* out, int lane) {
  __shared__ __attribute__((aligned(1024))) int32_t tile[640];
  const int32_t w = words[threadIdx.x], voff = 16 * threadIdx.x;
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(src), 0, 4096, 0x00020000);
  auto tracked = [&] {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)tile, 16, voff, 0, 0, 0);
  };
  tracked();
  const spr::i32x4_s desc = {__builtin_amdgcn_readlane(w, lane), __builtin_amdgcn_readlane(w, lane + 1),
                             __builtin_amdgcn_readlane(w, lane + 2), 0x00020000};
  const uint8_t* half = reinterpret_cast<uint8_t*>(tile + 256);
  spr::lds_dma16x2(desc, half, voff, desc, half + 512, voff + 512);
  tracked();
  spr::wait_vm<0>();
  spr::lds_barrier();
  out[threadIdx.x] = tile[threadIdx.x] + tile[256 + threadIdx.x];
}
"""


def test_inline_dma_states_what_it_reads_and_writes(tmp_path):
    """The DMA's asm block waits for a descriptor that a VALU instruction has just written (five
    wait states) and leaves m0 to the compiler, whose own DMA behind it relies on the base that it
    set before."""
    from sparsepr_amd import build_hip

    if shutil.which(build_hip.HIPCC) is None:
        pytest.skip("needs hipcc")
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(_DMA_PROBE)
    include = Path(build_hip.CSRC)
    subprocess.run([build_hip.HIPCC, *build_hip.FLAGS, "--cuda-device-only", "-S", f"-I{include}",
                    f"-I{include.parents[1] / 'include'}", str(src), "-o", str(asm)], check=True, capture_output=True)
    lines = [line.strip() for line in asm.read_text().splitlines()]
    lines = [line for line in lines if line.startswith((";;#ASM", "s_", "v_", "buffer_"))]
    dma = [i for i, line in enumerate(lines) if re.match(r"buffer_load_dword.* lds$", line)]
    assert len(dma) == 4, lines
    begin = max(i for i in range(dma[1]) if lines[i].startswith(";;#ASMSTART"))
    states = 0  # an instruction each, s_nop as many as it says
    for line in lines[begin + 1:dma[1]]:
        nop = re.match(r"s_nop (\d+)", line)
        states += int(nop.group(1)) + 1 if nop else 1
    assert states >= 5, lines[begin:dma[1] + 1]
    # m0 goes to a register before the DMA's base does into it, and comes back from there
    kept = re.match(r"s_mov_b32 (s\d+), m0$", lines[begin + 1])
    assert kept and f"s_mov_b32 m0, {kept.group(1)}" in lines[dma[2] + 1:dma[3]], lines[begin:dma[3] + 1]
    assert not any(re.search(rf"\b{kept.group(1)}\b", line) for line in lines[begin + 2:dma[2] + 1])


_ORDER_PROBE = """
#include <cstdio>
#include <cstdlib>
#include <hip/hip_runtime.h>
#include "spr_tile_order.h"
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3) {
    const spr::TileOrder o = spr::TileOrder::make(atoll(argv[i]), atoll(argv[i + 1]), atoll(argv[i + 2]));
    printf("%lld", static_cast<long long>(o.groups));
    for (int64_t b = 0; b < o.groups; ++b) {
      int64_t head;
      int32_t tile;
      o.at(static_cast<uint32_t>(b), head, tile);
      printf(" %lld %d", static_cast<long long>(head), tile);
    }
    printf("\\n");
  }
}
"""


def _tile_orders(tmp_path, calls):
    """Per (row tiles, most tiles, heads): the (head, tile) of each workgroup, [groups, 2]."""
    from sparsepr_amd import build_hip

    if shutil.which(build_hip.HIPCC) is None:
        pytest.skip("needs hipcc")
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(_ORDER_PROBE)
    subprocess.run([build_hip.HIPCC, "-std=c++17", "-O1", "-x", "hip", "--offload-host-only",
                    f"-I{build_hip.CSRC}", str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe), *(str(v) for call in calls for v in call)], check=True, capture_output=True)
    rows = [np.array(line.split(), dtype=np.int64) for line in out.stdout.decode().splitlines()]
    assert all(len(r) == 1 + 2 * r[0] for r in rows)
    return [r[1:].reshape(-1, 2) for r in rows]


def test_tile_order_deals_every_tile_once_and_the_longest_early(tmp_path):
    """Every tile of every head has one workgroup, with few to spare, and list scheduling on 8 XCDs
    of 32 workgroups ends near the ideal: with a prompt, whose query tiles keep every key and so walk
    1 / density = 5 times the chunks, and without one."""
    edges = [(rows, most, heads) for rows, most in ((1, 2), (7, 9), (16, 17), (31, 33), (32, 33), (79, 130), (127, 128), (128, 161),
                                                       (465, 765))
             for heads in (1, 2, 7, 8, 9, 24, 300)]
    for (rows, most, heads), order in zip(edges, _tile_orders(tmp_path, edges)):
        got = order[(order[:, 0] < heads) & (order[:, 1] < most)]
        assert len(got) == heads * most and len(np.unique(got, axis=0)) == heads * most
        run = 8 if rows >= 128 else 4 if rows >= 32 else 2
        assert len(order) <= heads * (most + 4 * run) + 16 * run  # two parts, each an odd number of runs
    rng = np.random.default_rng(0)
    cases = [(heads, tokens, text) for heads in (3, 5, 8, 12, 16, 24) for tokens in (20000, 35400, 60000, 118800)
             for text in (0, 256, 512)]
    calls = [(-(-(n + text) // 256), -(-(n + text) // 256) + n // 400, h) for h, n, text in cases]
    for (heads, tokens, text), call, order in zip(cases, calls, _tile_orders(tmp_path, calls)):
        ordinary = tokens // 5 // 64
        cost = np.zeros((heads, call[1]))
        for h in range(heads):
            live = -(-tokens // 256) + tokens // 800
            cost[h, :live] = np.sort(ordinary * rng.uniform(0.8, 1.1, live))[::-1]
            if text:
                cost[h, :live + 2] = np.concatenate(([5 * ordinary] * 2, cost[h, :live]))
        ends = np.zeros((8, 32))
        for b, (h, tile) in enumerate(order):
            if h < heads and tile < call[1]:
                xcd = ends[b % 8]
                xcd[xcd.argmin()] += cost[h, tile]
        # at most an ordinary tile and a half after the ideal end
        excess = (ends.max() - max(cost.sum() / 256, cost.max())) / ordinary
        assert excess <= 1.5, (heads, tokens, text, excess)
