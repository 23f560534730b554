// A group of lanes on the host: every lane is a context of its own, run one after another from one
// cross-lane operation to the next. Memory that the lanes share (a block's LDS, a group's global slot)
// is a list of regions of which every lane has a copy: a lane's stores reach the others at sync()
// alone, the point where the kernels order their memory operations (group_sync, clobber), so a
// missing one shows as an old value. Each region ends (or begins) at a page that may not be touched,
// and two lanes that store different values to one word between two sync() end the program.
#pragma once
#include <stdio.h>
#include <stdlib.h>
#include <sys/mman.h>
#include <ucontext.h>
#include <vector>

namespace emu {

struct Dim {
  unsigned x, y, z;
};
constexpr int kMaxLanes = 64;
extern int lanes, cur;  // group width, running lane
extern bool at_end;     // regions end at their guard page (else they begin at one)
extern unsigned char fill;

inline Dim thread_idx() { return {(unsigned)cur, 0, 0}; }
inline Dim block_dim() { return {(unsigned)lanes, 1, 1}; }
inline Dim one() { return {1, 1, 1}; }
inline Dim zero() { return {0, 0, 0}; }

inline unsigned char* guarded(size_t bytes) {
  const size_t page = 4096, body = (bytes + page - 1) / page * page;
  auto* p = (unsigned char*)mmap(nullptr, body + 2 * page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (p == MAP_FAILED || mprotect(p, page, PROT_NONE) || mprotect(p + page + body, page, PROT_NONE)) abort();
  unsigned char* q = p + page + (at_end ? body - bytes : 0);
  memset(q, fill, bytes);
  return q;
}

struct Region {
  size_t words = 0;
  bool uniform = false;          // every lane stores the same values (the control block)
  uint32_t* copy[kMaxLanes] = {};
  std::vector<uint32_t> base;
};
extern std::vector<Region*> regions;

template <class T>
T* region(Region& r, size_t count, bool uniform = false) {  // this lane's copy
  if (r.words == 0) {
    r.words = count * sizeof(T) / 4;
    r.uniform = uniform;
    for (int l = 0; l < lanes; ++l) r.copy[l] = (uint32_t*)guarded(count * sizeof(T));
    r.base.assign(r.copy[0], r.copy[0] + r.words);
    regions.push_back(&r);
  }
  return (T*)r.copy[cur];
}

void yield();                                    // to the next lane; back when all others have run
void meet(int kind);                             // every lane is at an operation of this kind
void sync();                                     // group_sync, clobber
uint64_t* box();                                 // a slot per lane for the values of one exchange

template <class T>
T from(int kind, T v, int src) {  // lane src's v (lanes past the group's read 0: inactive)
  uint64_t* b = box();
  uint64_t w = 0;
  memcpy(&w, &v, sizeof(T));
  b[cur] = w;
  meet(kind);
  T r{};
  if (src >= 0 && src < lanes) memcpy(&r, &b[src], sizeof(T));
  return r;
}

}  // namespace emu

template <class T>
T __shfl(T v, int src, int) { return emu::from(1, v, src); }
template <class T>
T __shfl_xor(T v, int m, int) { return emu::from(2, v, emu::cur ^ m); }
inline unsigned long long __ballot(bool p) {
  unsigned long long m = 0;
  uint64_t* b = emu::box();
  b[emu::cur] = p;
  emu::meet(3);
  for (int l = 0; l < emu::lanes; ++l) m |= (unsigned long long)b[l] << l;
  return m;
}
inline int __builtin_amdgcn_readlane(int v, int l) { return emu::from(4, v, l); }
inline int __builtin_amdgcn_readfirstlane(int v) { return emu::from(5, v, 0); }
inline int __builtin_amdgcn_ds_bpermute(int addr, int v) { return emu::from(6, v, addr / 4); }
inline int __builtin_amdgcn_mov_dpp(int v, int ctrl, int, int, bool) {
  const int l = emu::cur;
  int src = l;
  if (ctrl < 0x100) src = (l & ~3) | ((ctrl >> (2 * (l & 3))) & 3);  // quad_perm
  else if (ctrl == 0x140) src = (l & ~15) | (15 - (l & 15));         // row_mirror
  else if (ctrl == 0x141) src = (l & ~7) | (7 - (l & 7));            // row_half_mirror
  else abort();
  return emu::from(7, v, src);
}
struct Pair {
  int v[2];
  int operator[](int i) const { return v[i]; }
};
inline Pair __builtin_amdgcn_permlane16_swap(int a, int b, bool, bool) {  // odd rows of a <-> even rows of b
  const int b_even = emu::from(8, b, emu::cur & ~16), a_odd = emu::from(8, a, emu::cur | 16);
  const bool odd = emu::cur & 16;
  return {{odd ? b_even : a, odd ? b : a_odd}};
}
// inside divergent code, where the kernels ask only whether any lane takes a path that changes no other
inline unsigned long long __builtin_amdgcn_ballot_w64(bool p) { return p; }
inline int __double2loint(double v) {
  int64_t w;
  memcpy(&w, &v, 8);
  return (int)(uint32_t)w;
}
inline int __double2hiint(double v) {
  int64_t w;
  memcpy(&w, &v, 8);
  return (int)(w >> 32);
}
inline double __hiloint2double(int hi, int lo) {
  const uint64_t w = ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
  double v;
  memcpy(&v, &w, 8);
  return v;
}
template <class T, class U>
T atomicAdd(T* p, U v) {  // between lanes: one lane at a time
  const T o = *p;
  *p = o + (T)v;
  return o;
}
inline void __syncthreads() { emu::sync(); }
