"""The library's own choice of kernel for a call, from the host headers it compiles itself
(ellm_amd/csrc/*_plan.hpp), for tests that say which kernel their shapes reach.  256 compute units."""
import atexit
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ellm_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "general_plan.hpp"
#include "project_plan.hpp"
using namespace ellm;
static int project(char** v) {   // rows, heads, K
  uint32_t a[4];
  for (int i = 1; i <= 3; ++i) a[i] = (uint32_t)strtoul(v[i + 1], nullptr, 10);
  const proj::ProjectSplit s = proj::project_split(a[1], a[2], a[3], 256);
  printf("%u %u %zu %d\n", s.token_blocks, s.k_split, proj::split_floats(s, a[1], a[2]), (int)s.half_heads);
  return 0;
}
static int project_room(char** v) {   // heads, K, units, least and most rows of a handle: each one's room and what its calls' sums take at most
  uint32_t a[6];
  for (int i = 1; i <= 5; ++i) a[i] = (uint32_t)strtoul(v[i + 1], nullptr, 10);
  size_t need = 0;
  for (uint32_t rows = 1; rows <= a[5]; ++rows) {
    const size_t f = proj::split_floats(proj::project_split(rows, a[1], a[2], a[3]), rows, a[1]);
    need = f > need ? f : need;
    if (rows >= a[4]) printf("%zu %zu\n", proj::project_split_room(a[1], a[2], a[3], rows), need);
  }
  return 0;
}
static int project_block(char** v) {   // the workspace's floats, the room's, bytes that an allocation may have, status of a larger one
  const size_t most = strtoull(v[4], nullptr, 10);
  size_t part = strtoull(v[3], nullptr, 10);
  const int status = proj::project_block(strtoull(v[2], nullptr, 10), &part, [&](size_t bytes) {
    printf("%zu ", bytes);
    return bytes <= most ? 0 : atoi(v[5]);
  });
  printf("%zu %d\n", part, status);
  return 0;
}
static int chunk(char** v) {   // batch capacity, batch, query heads, key-value heads, most positions a call, position_index, interval, bfloat16
  uint32_t a[9];
  for (int i = 1; i <= 8; ++i) a[i] = (uint32_t)strtoul(v[i + 1], nullptr, 10);
  const ChunkCall c = {a[6], a[7], a[2], a[1], a[3], a[4], 256, prefill_workspace_rows(a[5], a[1], a[3], 256), a[8] != 0};
  const ChunkPlan p = plan_chunk(c);
  printf("%d %u %u %u %d %u\n", (int)p.kernel, p.kernel == kChunkStream ? p.waves : p.kernel == kChunkShort ? p.row_blocks : 0, p.n_split, p.n_wg,
         (int)p.form, p.split_tiles * kChunkTile);
  return 0;
}
// head size, bytes an element, batch capacity, batch, query heads, key-value heads, most positions a call,
// position_index, interval, whole aligned pieces, and room for partial rows per query row (0: the workspace's)
int main(int, char** v) {
  if (v[1][0] == 'c') return chunk(v);
  if (v[1][0] == 'p') return project(v);
  if (v[1][0] == 'r') return project_room(v);
  if (v[1][0] == 'b') return project_block(v);
  uint32_t a[12];
  for (int i = 1; i <= 11; ++i) a[i] = (uint32_t)strtoul(v[i], nullptr, 10);
  const gen::GeneralWorkspace w = gen::general_workspace(a[7], a[3], a[5], a[6], a[1], 256);
  gen::GeneralCall c;
  c.planes = a[4] * a[6];
  c.group = a[5] / a[6];
  c.interval = a[9];
  c.max_len = a[8] + a[9];
  c.n_cu = 256;
  c.head_size = a[1];
  c.f32 = a[2] == 4;
  c.vec = a[10] != 0;
  c.room = a[11] ? a[11] : w.rows / (c.planes * c.rows());
  const gen::GeneralPlan p = gen::general_plan(c);
  printf("%d %u %u %u %d %zu %d %u\n", (int)p.kernel, p.n_split, p.tile_rows, p.key_groups, p.nb, w.rows, (int)p.max_first, p.split_len);
}
"""


@functools.lru_cache(maxsize=None)
def _program():
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    d = tempfile.mkdtemp(prefix="plan_probe_")
    atexit.register(shutil.rmtree, d, True)
    with open(os.path.join(d, "probe.cpp"), "w") as f:
        f.write(SOURCE)
    exe = os.path.join(d, "probe")
    subprocess.run([gxx, "-O1", "-std=c++17", "-I", CSRC, "-o", exe, os.path.join(d, "probe.cpp")], check=True)
    return exe


def general_plan(head_size, element_bytes, batch_capacity, batch, q_heads, kv_heads, position_index, interval, vec=None, room=0):
    """(kernel "rows" / "step" / "chunk", key splits, rows per workgroup, key groups, padded head blocks, the
    workspace's partial rows, whether a chunk kernel looks for the row maximum every step, keys a split)"""
    if vec is None:
        vec = head_size * element_bytes % 16 == 0
    args = (head_size, element_bytes, batch_capacity, batch, q_heads, kv_heads, interval, position_index, interval, int(vec), room)
    out = subprocess.run([_program(), *map(str, args)], check=True, capture_output=True, text=True).stdout.split()
    return (("rows", "step", "chunk")[int(out[0])], *map(int, out[1:]))


def project_split(rows, heads, k):
    """Projection of 65 rows and more: (128-token blocks a tile, workgroups that share its K, their sums' floats,
    whether eight waves of half a head walk a tile)"""
    out = subprocess.run([_program(), "p", *map(str, (rows, heads, k))], check=True, capture_output=True, text=True)
    return tuple(map(int, out.stdout.split()))


def project_room(heads, k, least, most, units=256):
    """[(a handle's room, the most that the sums of any of its calls take)] for handles of `least` .. `most` rows"""
    out = subprocess.run([_program(), "r", *map(str, (heads, k, units, least, most))], check=True, capture_output=True, text=True)
    return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]


def project_block(ws, part, most, status):
    """A handle's block where allocations beyond `most` bytes end with `status`: (bytes asked for in turn, the room it got
    in floats, the last status)"""
    out = subprocess.run([_program(), "b", *map(str, (ws, part, most, status))], check=True, capture_output=True, text=True)
    *asked, room, last = map(int, out.stdout.split())
    return asked, room, last


def _chunk(batch_capacity, batch, q_heads, kv_heads, position_index, interval, most=None, bf16=False):
    args = ("c", batch_capacity, batch, q_heads, kv_heads, most or interval, position_index, interval, int(bf16))
    return subprocess.run([_program(), *map(str, args)], check=True, capture_output=True, text=True).stdout.split()


def chunk_plan(*call, **most):
    """128-wide 16-bit heads: (kernel "stream" / "pingpong" / "short", its waves or row blocks, key splits, workgroups a split).
    Arguments: batch capacity, batch, query heads, key-value heads, position_index, interval[, most positions a call]"""
    out = _chunk(*call, **most)
    return (("stream", "pingpong", "short")[int(out[0])], *map(int, out[1:4]))


def chunk_form(*call, **more):
    """The form of the tile kernel that an unsplit call of it runs: "registers", "direct" or "wide"; for the last one
    the storage type counts (bf16=True)."""
    return ("registers", "direct", "wide")[int(_chunk(*call, **more)[4])]


def chunk_piece_keys(*call, **more):
    """Keys a piece of a split call."""
    return int(_chunk(*call, **more)[5])


def chunk_is_direct(*call, **more):
    return chunk_form(*call, **more) == "direct"
