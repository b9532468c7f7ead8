// The order in which a block comes to the pairs of its groups of centres (basis_group.hip).  Host
// code as well: a walk is whole numbers only and can be followed on the CPU.
#pragma once
#include "common.h"

namespace mccnn {

// The centres of a group that have pairs, from its first place in the order on (in a group without
// pairs one centre of none).
struct __align__(16) GroupCentre {
  int centre, begin, count;           // its pairs
  int flags;                          // 1: the group's last, 2: GroupInfo::direct, 4 x GroupInfo::rows
};

struct GroupChunk {
  int centre, begin, left;            // left: pairs of the centre from begin on
  int group;                          // its group, or -1 past the last chunk
  int rows, direct;                   // of the group
  int odd;                            // which of two buffers holds the group's keys
  bool first, last;                   // of the group
};

// The same value in every lane, where the compiler cannot see it.
__host__ __device__ __forceinline__ int same_in_all(int x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_readfirstlane(x);
#else
  return x;
#endif
}

// Walks the groups first_group, first_group + stride, ..  below `groups`, of `group` places each,
// in chunks of up to kChunk pairs of one centre.  The centre after the one being read is fetched by
// every lane and looked at in the next read().
template <int kChunk>
struct GroupWalk {
  const GroupCentre *listed;
  int64_t n_out;                      // centres
  int group, groups, stride;
  int at_group;                       // group of the centre after the one being read
  int64_t at;                         // and its place
  GroupCentre after = {0, 0, 0, 1};
  int centre = 0, begin = 0, left = 0, flags = 0, group_read = 0, odd = 0;
  bool fresh = true;                  // the next centre starts a group

  __host__ __device__ __forceinline__ GroupWalk(const GroupCentre *listed, int64_t n_out, int group,
                                                int groups, int stride, int first_group)
      : listed(listed), n_out(n_out), group(group), groups(groups), stride(stride),
        at_group(first_group), at((int64_t)first_group * group) {}

  __host__ __device__ __forceinline__ void fetch() {
    int64_t place = at < n_out ? at : n_out - 1;
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(place));   // (a vector load, though the same for all lanes)
#endif
    after = listed[place];
  }

  // The next chunk; fetch() goes before every call.
  __host__ __device__ __forceinline__ GroupChunk read() {
    GroupChunk c{0, 0, 0, -1, 0, 0, 0, false, false};
    while (left <= 0) {               // the next centre (twice: groups without pairs)
      if (at_group >= groups) return c;
      centre = same_in_all(after.centre);
      begin = same_in_all(after.begin);
      left = same_in_all(after.count);
      flags = same_in_all(after.flags);
      group_read = at_group;
      if (fresh) c.first = true;
      fresh = flags & 1;
      at = fresh ? (int64_t)(at_group += stride) * group : at + 1;
      if (left <= 0) fetch();
    }
    // Groups without pairs leave the buffers as they are: the keys of the group before this one are
    // still to be read when its own are stored.
    if (c.first) odd ^= 1;
    c.centre = centre;
    c.begin = begin;
    c.left = left;
    c.group = group_read;
    c.rows = flags >> 2;
    c.direct = flags & 2;
    c.odd = odd;
    begin += kChunk;
    left -= kChunk;
    c.last = left <= 0 && (flags & 1);
    return c;
  }
};

}  // namespace mccnn
