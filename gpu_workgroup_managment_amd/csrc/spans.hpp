// spans.hpp -- positions in a graph's arrays (no HIP in it: constexpr functions
// serve host and device).
//
// A graph may have 2^31 - 1 edges and as many vertices, and a loop steps by
// lanes, workgroups or grids: as a signed 32-bit index it would step past 2^31
// before it compares, come out negative and go on. Positions are unsigned here:
// a step of less than 2^31 past the last one does not wrap, at the same cost.
#pragma once

#include <cstdint>

namespace wgm {

// What is left of the positions [first, stop).
struct Span {
  uint32_t at, stop;
  // Whether the position k after the current one is among them.
  constexpr bool has(uint32_t k = 0) const { return at + k < stop; }
  constexpr void next(uint32_t step) { at += step; }
  // The end of at most k positions from the current one on.
  constexpr uint32_t until(uint32_t k) const { return at + k < stop ? at + k : stop; }
};

// A search for a position in [a, b] by rounds of 64 probes, evenly spaced: the
// answer is past every probe that is below it, and the probes below it come first.
struct Split {
  uint32_t a, b;
  constexpr bool open() const { return a < b; }
  constexpr uint32_t step() const { return (b - a + 63u) >> 6; }
  constexpr uint32_t probe(uint32_t lane) const { return a + lane * step(); }
  // The first k probes (k > 0) are below the answer.
  constexpr void narrow(uint32_t k) {
    const uint32_t last = probe(k - 1u), next = last + step();
    b = next < b ? next : b;
    a = last + 1u;
  }
};

}  // namespace wgm
