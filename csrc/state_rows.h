// How the 256 threads of the kernels for single tokens share a head's state [rows][width] (floats; width a multiple of 4, at most 1024): a thread has four columns
// of the rows group, group + groups, ...  Without branches around its loads it reads at first, first + stride, ... as often as the kernel has registers for, behind
// its last row at `first` again; a thread without rows (columns that do not fill the threads, or more groups than rows) reads the head's first floats.
#pragma once

struct StateRows {
  int group, groups, col;  // group >= groups: no columns
  int first, stride;       // offset of the thread's first float of four, and from one of its rows to the next
  int count;               // rows
  __host__ __device__ bool on() const { return group < groups; }
  __host__ __device__ int at(int i) const { return first + (i < count ? i * stride : 0); }  // of its row i
};

__host__ __device__ inline StateRows state_rows(int tid, int rows, int width) {
  StateRows s;
  const int chunks = width >> 2;
  s.groups = 256 / chunks;
  s.group = tid / chunks;
  s.col = (tid - s.group * chunks) * 4;
  s.stride = s.groups * width;
  s.count = s.on() && s.group < rows ? (rows - s.group + s.groups - 1) / s.groups : 0;
  s.first = s.count ? s.group * width + s.col : 0;
  return s;
}
