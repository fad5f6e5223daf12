// Which item a workgroup of a chain of dependent steps executes next (encoder_chain.hip, decoder_chain.hip).  Plain arithmetic, so that a test can
// drive it without a device.
//
// A workgroup takes every G-th item of each step.  One that has waited in vain for what an item reads executes the steps that it misses by
// itself, from one whose inputs it has seen (`solo`), and goes on with the item.  It does so once for an item: then everything the item reads has
// been written, by itself if by nobody else, and is at most in flight.  Who still waits has met a mistake in a shape or a rule, and gives up
// after kChainMostTries rounds of waiting, so that the launch ends whatever a mistake there may be: at most one pass over the steps and kChainMostTries
// rounds for each of its items.
#pragma once

#include <cstdint>

#if defined(__HIP__)
#define TTMI_WALK __host__ __device__ __forceinline__
#else
#define TTMI_WALK inline
#endif

namespace ttmi {

constexpr int kChainMostTries = 4096;

// Launches whose order the host does not know are counted in memory, in units that the workgroups of each add up between them, one share when each ends.
// While one has not ended a unit is not full, so that whoever reads the count, however late it started, finds the same number of whole units.
constexpr uint32_t kLaunchUnit = 1u << 16;
constexpr int kChainMostWorkgroups = 1 << 15;  // (a share of at least one, in 32 bits)
TTMI_WALK uint32_t launch_share(uint32_t rank, uint32_t workgroups) { return (rank + 1) * kLaunchUnit / workgroups - rank * kLaunchUnit / workgroups; }

struct ChainWalk {
  int step = 0, item = 0;                // the item at hand
  int resume_step = 0, resume_item = 0;  // while solo: the one that waits
  int tries = 0;                         // rounds of waiting for the item at hand
  int pass = 0;                          // of the item that the workgroup was given: 0 none, 1 on it (solo), 2 over

  TTMI_WALK bool solo() const { return pass == 1; }
  // The first item at or behind (step, item + stride) of those that the workgroup is given.
  template <typename Items, typename First>
  TTMI_WALK void forward(int stride, int end, const Items& items, const First& first_item) {
    item += stride;
    while (step < end && item >= items(step)) {
      ++step;
      if (step < end) item = first_item(step);
    }
  }
  // The item at hand has been executed; the chain is done for the workgroup once step == end.
  template <typename Items, typename First>
  TTMI_WALK void executed(int stride, int end, const Items& items, const First& first_item) {
    tries = 0;
    if (pass != 1) {
      pass = 0;
      forward(stride, end, items, first_item);
    } else if (++item >= items(step)) {
      item = 0;
      if (++step == resume_step) item = resume_item, pass = 2;
    }
  }
  // What the item at hand reads is not there; the inputs of step `from` are.  false: nor will it be.
  TTMI_WALK bool late(int from) {
    if (pass == 0 && from < step) {
      pass = 1;
      resume_step = step, resume_item = item;
      step = from, item = 0;
      tries = 0;
      return true;
    }
    return ++tries <= kChainMostTries;
  }
};

}  // namespace ttmi
