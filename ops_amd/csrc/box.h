// Copies of point boxes between pitched device arrays and dense host memory.
#pragma once

#include "runtime.h"

namespace opsmi {

// planes x rows x width bytes; comps > 1: the array keeps each component of
// elem bytes cstride bytes apart (structure of arrays), the host buffer a
// point's components together, and width counts all components
struct Box {
  char *base;          // first point
  long pitch, plane;   // bytes between rows and planes
  size_t width;        // bytes per row of the box
  unsigned rows, planes;
  unsigned comps = 1, elem = 1;
  long cstride = 0;
};

// box <-> buf (ordinary host memory), on stream s; returns when buf (or the
// array) holds the values
void box_copy(Staging &st, hipStream_t s, Box b, char *buf, bool to_device);

// dst = src outside the points of r, both whole arrays laid out as d's (one
// array: not structure of arrays), on the library's stream
void copy_outside(ops_dat d, char *dst, const char *src, const Range3 &r);

// whether a caller's buffer is device memory (fetch and set take either kind)
bool device_pointer(const void *p);

}  // namespace opsmi
