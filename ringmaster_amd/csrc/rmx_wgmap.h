// Workgroup placement of the attention kernels, host and device.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/ringmaster_amd.h"

namespace rmx {

// ---------------------------------------------------------------------------
// Workgroup -> (problem, group, tile) mapping shared by the attention kernels.
// A "group" is one (batch, head) of a problem (its tiles share K/V or Q/dO) and
// every group has ntile[p] workgroups. Problems are ordered longest-workgroup
// first by the launcher. Balanced mode (every problem's group count divisible
// by 8): the dispatcher deals workgroup ids round-robin over the 8 XCDs, so
// XCD x = bid % 8 runs ids bid = 8 i + x in order of i, and each XCD gets an
// eighth of every problem's groups (one XCD's L2 serves a group's shared
// operand): q heads of one KV head together when the KV heads divide by 8
// (share > 1: their K/V is then read into one L2 instead of up to `share`),
// else groups g with g % 8 == x.
// Inside an XCD's part of a problem the order is group by group, a group's tiles
// longest first. Causal tiles differ in length, and the last group started is then
// a long one beside idle CUs when an XCD runs only a few groups of few tiles: with
// 4 groups of 16 tiles on 32 CUs the last CU ends after 100 tile steps against 68
// for an even share. There `set` groups run tile by tile across the set (68 steps).
struct WgMapParams {
  int nprob;
  int balanced;
  int share;                       // balanced: q heads per KV head kept on one XCD (1: off)
  int set;                         // groups interleaved tile by tile
  int ngroup;                      // groups per problem (balanced: per problem and XCD)
  int ntile[RMX_MAX_BATCHED];
  int start[RMX_MAX_BATCHED + 1];  // balanced: per-XCD prefix; else: global prefix
  int total;                       // workgroups doing work (grid may be larger)
};

struct WgCoord {
  int p, group, tile;
  bool valid;
};

__host__ __device__ __forceinline__ WgCoord map_workgroup(const WgMapParams& m, int bid) {
  WgCoord c;
  const int i = m.balanced ? (bid >> 3) : bid;
  c.valid = m.balanced ? (i < m.start[m.nprob]) : (bid < m.total);
  int p = 0;
  while (p + 1 < m.nprob && i >= m.start[p + 1]) ++p;
  const int local = i - m.start[p], nt = m.ntile[p];
  c.p = p;
  int g;  // group among the XCD's (or all) groups
  if (m.set > 1) {
    const int first = local / (m.set * nt) * m.set;
    const int gs = m.ngroup - first < m.set ? m.ngroup - first : m.set;
    const int r = local - first * nt;
    c.tile = r / gs;
    g = first + r % gs;
  } else {
    c.tile = local % nt;
    g = local / nt;
  }
  const int x = bid & 7;
  c.group = !m.balanced ? g : m.share > 1 ? ((g / m.share) * 8 + x) * m.share + g % m.share : g * 8 + x;
  return c;
}

// Host side: fill the mapping for problems already in launch order; groups = groups of every
// problem, share = consecutive groups that read the same K/V (q heads of one KV head),
// ntile[p] = workgroups per group, uneven = a group's tiles differ in length (causal masks).
// Returns the grid size.
inline int plan_workgroups(WgMapParams& m, int n, int groups, int share, const int* ntile,
                           bool uneven) {
  m.nprob = n;
  m.balanced = n > 0 && groups % 8 == 0;
  m.share = m.balanced && (groups / share) % 8 == 0 ? share : 1;
  m.ngroup = m.balanced ? groups / 8 : groups;
  int acc = 0, most = 1;
  for (int i = 0; i < n; ++i) {
    m.ntile[i] = ntile[i] > 0 ? ntile[i] : 1;
    m.start[i] = acc;
    acc += m.ngroup * (ntile[i] > 0 ? ntile[i] : 0);
    most = ntile[i] > most ? ntile[i] : most;
  }
  for (int i = n; i <= RMX_MAX_BATCHED; ++i) m.start[i] = acc;
  m.total = acc;
  // Two rounds of workgroups per XCD (64 on 32 CUs; unbalanced: 512 on 256) make an even share
  // out of one set; longer groups are even by themselves.
  const int round = m.balanced ? 32 : 256;
  m.set = uneven && most < round ? (2 * round + most - 1) / most : 1;
  return m.balanced ? 8 * acc : acc;
}

}  // namespace rmx
