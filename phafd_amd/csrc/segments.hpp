// segments.hpp -- walks over the slots [s, e) of a pair list, e up to 2^31 - 1.
//
// Slots are ints; a walk that takes several at a time steps past e, and near
// the largest list past the type.  Both walks are constant expressions, so an
// overflow in them is a compile error where they are tried at the limit.
#pragma once
#if defined(__HIPCC__)
#define PHAFD_SEG __host__ __device__ __forceinline__ constexpr
#else
#define PHAFD_SEG constexpr
#endif

namespace phafd {

// one lane's slots: s + lane and every G-th after it (unsigned: the step past e fits)
struct LaneWalk {
  unsigned c, e;
  PHAFD_SEG LaneWalk(int s, int end, int lane) : c((unsigned)s + (unsigned)lane), e((unsigned)end) {}
  PHAFD_SEG bool on() const { return c < e; }
  PHAFD_SEG void next(int G) { c += (unsigned)G; }
};

// the end of a chunk of at most `most` slots from c, which is where the next one starts
PHAFD_SEG int chunk_end(int c, int e, int most) { return e - c > most ? c + most : e; }

}  // namespace phafd
