// The workgroup -> (batch, q-head, row block) schedule of the 16-bit prefill kernel
// (fa_prefill.hip), kept apart from the kernel body.
#pragma once

#include <algorithm>

#include "fa_device.hpp"
#include "fa_internal.hpp"

namespace fa {

struct PrefillItem {
  int b;    // batch (varlen: sequence)
  int hq;   // q-head
  int kvh;  // kv-head
  int rb;   // row block (NW * rows-per-wave queries)
};

// Workgroup blockIdx.x -> work item; false for grid padding (varlen), uniform over the workgroup.
//
// Dense: scheduling units are the q-heads of as many kv-heads as keep about unit_bytes of
// K/V (prefill_unit_bytes; one XCD's L2 is 4 MB).  Units follow each other in logical order, and
// each XCD gets a contiguous range of it, so an XCD works through one
// or two units at a time and re-reads K/V from its L2.  Inside a unit the query blocks go by
// rank, heaviest causal blocks first, all heads of the unit at each rank, which keeps the
// XCD's CUs evenly loaded to the end.
//
// Varlen: sequences differ in length, and ranges of whole sequences per XCD load the XCDs
// unevenly (measured: a 16-sequence batch ran at 0.18 of peak).  There the order is
// rank-major per XCD: the dispatcher deals workgroups to the XCDs round-robin (blockIdx % 8),
// XCD x takes the (sequence, kv-head) groups g = x (mod 8) and walks them rank by rank,
// heaviest causal ranks first, with the q-heads of one kv-head side by side, so they run
// together and read its K/V through one L2 (measured: +8-10% over rank-major across all
// XCDs, which fetched each K/V tile into up to four L2s).  The host pads the grid to a
// multiple of 8 groups; padding returns false.

// K/V bytes of the q-heads one dense scheduling unit holds.  At D=128 half an XCD's L2: the
// Q and O streams (64 KiB each per 256-row workgroup) pass through the same L2, and a unit
// whose K/V filled all 4 MB had them evicted and re-fetched (causal GQA B=4 Hq=32 Hkv=8 N=4096:
// 296 MB read for 201 MB of Q, K and V with 4 MB units, 216 MB with 2 MB units, at the same
// speed).  At D <= 64 a workgroup's Q and O are half as large or less, and halving the unit
// cost 2-8% (MHA D=64 N=4096: fewer heads to spread over the XCD's CUs), so those keep 4 MB.
inline int64_t prefill_unit_bytes(int head_dim) { return int64_t{head_dim == 128 ? 2 : 4} << 20; }

// The q-heads of as many whole kv-heads as fit prefill_unit_bytes: the most a dense scheduling unit holds.
inline int prefill_unit_heads(int nk, int head_dim, int group) {
  const int64_t kv_head_bytes = (int64_t)(nk > 1 ? nk : 1) * head_dim * 2 * 2;
  const int64_t kv_heads = prefill_unit_bytes(head_dim) / kv_head_bytes;
  return (int)(kv_heads > 1 ? kv_heads : 1) * group;
}

// Causal: an XCD's range must start with its heaviest blocks and end with its lightest.  A unit cut by a
// range's end leaves ranks 16-9 on one XCD and 8-1 on the next (the prompt of one request, Hq=32 Hkv=8
// N=1999, 8-head units: 1.47 times the mean load), or the heaviest blocks of the next unit to an XCD's last
// round (D=128 B=7 Hq=16 Hkv=4 N=600, 24-head units 29.4 us, 12-head units 35.3, an XCD's own 14 heads 26.2).
// Where the heads divide by the 8 XCDs each XCD therefore takes its share of them in units of its own: as few
// as keep to prefill_unit_heads, of nearly equal size.  B=9 Hq=8 Hkv=1 N=1100 46.1 -> 38.7 us, B=3 Hq=16
// Hkv=4 N=1500 50.0 -> 41.0, B=8 Hq=32 Hkv=8 N=700 64.1 -> 60.2.
// q-heads of one XCD, 0 where the XCDs' ranges do not hold whole heads (or need not: without the causal mask)
inline int prefill_share(bool causal, int64_t heads) { return causal && heads % 8 == 0 ? (int)(heads / 8) : 0; }
// Heads that do not divide are dealt to the XCDs rank by rank where that beats one order over all heads: grids
// of more than one workgroup per CU, with fewer than 32 heads or D <= 64 (D=64 B=7 Hq=12 N=1500 49.1 -> 38.6
// us; 25 heads N=1300 D=128 35.5 -> 27.5).  Dealt, every XCD reads every K/V: with more heads at D >= 128 that
// can cost what the balance gains (B=9 Hq=12 Hkv=4 N=1500, D=128 94.8 -> 86.6, D=256 176 -> 187), and so it
// does where the first row block sees more than half of what the last one sees (D=64 B=7 Hq=20, 178 queries on
// 565 keys 18.0 -> 19.7).
inline bool prefill_deal(bool causal, int64_t heads, int64_t total, int head_dim, int nq, int nk) {
  return causal && heads % 8 != 0 && total > 256 && (heads < 32 || head_dim <= 64) && 2 * ((int64_t)nk - nq + 128) <= nk;
}
inline int64_t prefill_units(bool causal, int64_t heads, int group, int nk, int head_dim) {
  const int64_t most = std::min<int64_t>(prefill_unit_heads(nk, head_dim, group), heads);
  const int64_t share = prefill_share(causal, heads);
  if (share == 0) return most;
  if (share <= most) return share;
  const int64_t units = (share + most - 1) / most, even = (share + units - 1) / units;
  return (even + group - 1) / group * group;  // whole kv-heads: at most `most`, itself a multiple of group
}

// The schedule fields of a dense call's arguments (kv_groups, group, nq, nk, causal, n_rowblk and total are set;
// nw: waves per workgroup).
inline void prefill_schedule(TileArgs& a, int head_dim, int nw) {
  const bool causal = a.causal != 0;
  const int64_t heads = (int64_t)a.kv_groups * a.group;
  a.deal = prefill_deal(causal, heads, a.total, head_dim, a.nq, a.nk);
  a.share = prefill_share(causal, heads);
  // at most `heads`, so that u_items <= total
  a.u_heads = (int32_t)(a.deal ? heads : prefill_units(causal, heads, a.group, a.nk, head_dim));
  a.u_items = a.u_heads * a.n_rowblk;
  // (in one order over all heads a range starts anywhere in a unit: reversed, B=3 Hq=12 Hkv=4 N=1000 D=128
  // 26.8 -> 29.8 us)
  a.fold = causal && (a.deal || a.share > 0) && nw == 4 && head_dim <= 128 && a.total > 256 && a.total <= 512;
}

struct PrefillOrder {
  uint32_t rank, head;  // head: (batch, q-head) pair
};

// Workgroup -> rank and head of a dense call.  Every quantity is non-negative: unsigned division needs no
// sign fix-ups, and all waves of the workgroup run this scalar code before their first DMA.
__host__ __device__ inline PrefillOrder prefill_dense_order(const TileArgs& a, uint32_t bid) {
  constexpr uint32_t kXcds = 8;
  // a.fold: the grid fits the GPU at two workgroups per CU.  The dispatcher gives each of an XCD's 32
  // CUs one workgroup and then a second, so the first 32 are taken in reverse: the CU with the heaviest
  // of them gets the lightest of the rest (in order, the heaviest would get the heaviest again).
  // With units cut to an XCD's share, Hq=32 Hkv=8 N=1999 causal D=128: 54.5 -> 45.6 us; 16 heads,
  // N=4000: 97.8 -> 77.0.
  uint32_t slot = bid / kXcds;
  if (a.fold && slot < 32) slot = 31 - slot;
  const uint32_t xcd = bid % kXcds, pid = slot * kXcds + xcd;
  // the XCD's own heads (prefill_share), or one order over all heads: dealt to the XCDs one by one
  // (a.deal), or a contiguous range each
  const uint32_t heads = a.share > 0 ? (uint32_t)a.share : (uint32_t)a.kv_groups * (uint32_t)a.group;
  const uint32_t first = xcd * (uint32_t)a.share;
  const uint32_t logical = a.share > 0 ? slot : a.deal ? pid : (uint32_t)xcd_remap((int)pid, a.total);
  const uint32_t unit = logical / (uint32_t)a.u_items;
  const uint32_t within = logical - unit * (uint32_t)a.u_items;
  const uint32_t left = heads - unit * (uint32_t)a.u_heads;
  const uint32_t unit_size = left < (uint32_t)a.u_heads ? left : (uint32_t)a.u_heads;
  const uint32_t rank = within / unit_size;
  return {rank, first + unit * (uint32_t)a.u_heads + (within - rank * unit_size)};
}

template <int D>
__device__ __forceinline__ bool prefill_item(const TileArgs& a, PrefillItem& it) {
  constexpr uint32_t kXcds = 8;
  const uint32_t group = (uint32_t)a.group, bid = blockIdx.x;
  uint32_t mrev, item;
  if (a.varlen) {
    const uint32_t xcd = bid % kXcds, local = bid / kXcds;
    const uint32_t per_rank = (uint32_t)a.total / ((uint32_t)a.n_rowblk * kXcds);  // this XCD's items per rank
    mrev = local / per_rank;
    const uint32_t j = local - mrev * per_rank;
    const uint32_t jg = j / group;
    const uint32_t kvg = jg * kXcds + xcd;
    if (kvg >= (uint32_t)a.kv_groups) return false;
    item = kvg * group + (j - jg * group);
  } else {
    const PrefillOrder o = prefill_dense_order(a, bid);
    mrev = o.rank;
    item = o.head;
  }
  const uint32_t kvi = item / group;
  const uint32_t gi = item - kvi * group;
  const uint32_t bb = kvi / (uint32_t)a.hkv;
  it.kvh = (int)(kvi - bb * (uint32_t)a.hkv);
  it.b = (int)bb;
  it.hq = it.kvh * a.group + (int)gi;
  it.rb = a.causal ? (a.n_rowblk - 1 - (int)mrev) : (int)mrev;  // heaviest causal blocks first
  return true;
}

}  // namespace fa
