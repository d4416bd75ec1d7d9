// Launch classes of the FTL step: (points per lane M, lanes per strand G,
// guarded).  Exact classes need npoints == M * G; guarded classes accept any
// npoints <= M (G = 1) or (G - 1) * M < npoints <= G * M (G = 2 or 4).  The class id indexes the per-class kernels and the
// `cls` field of batched tiles.
#pragma once

// X(id, points per lane, lanes per strand, guarded, waves per SIMD targeted
// by the register allocator: the highest at which neither the plain nor the
// tile-list kernel of the class spills to memory (1 and 11 fit six, where they
// hold one row of loads in flight instead of three: us a step, six and five, 134
// MB of 8 points 68.5, 52.7, in wind 69.2, 66.1; of 7 76.9, 65.3, in wind 75.8,
// 76.6), points per lane of a load/store
// chunk: 8 float4 make one 128-byte line, so each line of the groom is read
// by one request; 4 halves the LDS stage where a bigger one would cost
// occupancy, at the price of two requests per line)
#define FTL_CLASSES(X)        \
  X(0, 4, 1, false, 8, 4)     \
  X(1, 8, 1, false, 5, 4)     \
  X(2, 16, 1, false, 4, 4)    \
  X(3, 32, 1, false, 2, 8)    \
  X(4, 8, 2, false, 4, 8)     \
  X(5, 16, 2, false, 4, 8)    \
  X(6, 32, 2, false, 2, 8)    \
  X(7, 4, 4, false, 6, 4)     \
  X(8, 8, 4, false, 4, 8)     \
  X(9, 16, 4, false, 4, 8)    \
  X(10, 4, 1, true, 6, 4)     \
  X(11, 8, 1, true, 5, 4)     \
  X(12, 16, 1, true, 4, 4)    \
  X(13, 32, 1, true, 2, 4)    \
  X(14, 64, 1, true, 1, 8)    \
  X(15, 4, 2, false, 7, 4)     \
  X(16, 48, 1, true, 1, 8)     \
  X(17, 8, 2, true, 4, 8)      \
  X(18, 16, 2, true, 2, 8)     \
  X(19, 32, 2, true, 2, 8)     \
  X(20, 12, 2, true, 4, 4)     \
  X(21, 24, 2, true, 3, 8)     \
  X(22, 16, 4, true, 3, 8)     \
  FTL_VARIANTS(X)

// Tile-shape variants of exact classes: the same (M, G) with another load /
// store chunk or occupancy target.  ftl_class_for never picks them on its
// own; the autotuner times them beside the base classes and its tables
// select them per point count.
#define FTL_VARIANTS(X)        \
  X(23, 16, 2, false, 2, 4)    \
  X(24, 16, 4, false, 3, 4)    \
  X(25, 8, 2, false, 4, 4)     \
  X(26, 8, 4, false, 6, 8)     \
  X(27, 32, 1, false, 2, 4)    \
  X(28, 16, 1, false, 3, 4)

#define FTL_NCLASSES 29

struct FtlClassInfo {
  int m, g, guarded, waves, chunk;
};

static constexpr FtlClassInfo kFtlClasses[FTL_NCLASSES] = {
#define FTL_CI(id, M, G, GU, W, CH) {M, G, GU ? 1 : 0, W, CH},
    FTL_CLASSES(FTL_CI)
#undef FTL_CI
};

// Load/store chunk of a tile of M points per lane.  A kernel translation unit
// compiles one class (FTL_CLASS_ID), whose chunk it takes; elsewhere, the
// first class with these parameters.
constexpr int ftl_chunk_of(int m, int g, bool guarded) {
#ifdef FTL_CLASS_ID
  (void)g;
  (void)guarded;
  return kFtlClasses[FTL_CLASS_ID].chunk < m ? kFtlClasses[FTL_CLASS_ID].chunk : m;
#else
  for (int i = 0; i < FTL_NCLASSES; ++i)
    if (kFtlClasses[i].m == m && kFtlClasses[i].g == g && (kFtlClasses[i].guarded != 0) == guarded)
      return kFtlClasses[i].chunk < m ? kFtlClasses[i].chunk : m;
  return m < 4 ? m : 4;
#endif
}

// Wide forms (ftl_wide.h): X(points per lane M, lanes per strand G); a form
// takes any point count N with M = ceil(N / G).  Not launch classes: the
// library picks them by the size of a launch (ftl_wide_level, ftl_wide_form).
// FTL_LEVEL_FORMS: only in launches smaller than the chip, whose state of at most
// 16 waves a CU, 64 MB on 256 CUs, is always written through.
// FTL_DEFAULT_FORMS: also in launches that fill it.
#define FTL_LEVEL_FORMS_2(X)
#define FTL_LEVEL_FORMS_4(X) X(1, 4) X(2, 4) X(3, 4) X(4, 4)
#define FTL_LEVEL_FORMS_8(X) X(1, 8) X(2, 8) X(3, 8) X(4, 8)
#define FTL_LEVEL_FORMS_16(X) X(1, 16) X(2, 16) X(3, 16) X(4, 16)
#define FTL_DEFAULT_FORMS_2(X) X(3, 2) X(4, 2) X(5, 2) X(6, 2) X(7, 2) X(8, 2)
#define FTL_DEFAULT_FORMS_4(X) X(5, 4) X(6, 4) X(7, 4) X(8, 4)
#define FTL_DEFAULT_FORMS_8(X) X(5, 8) X(6, 8) X(7, 8) X(8, 8)
#define FTL_DEFAULT_FORMS_16(X)
#define FTL_DEFAULT_FORMS(X) FTL_DEFAULT_FORMS_2(X) FTL_DEFAULT_FORMS_4(X) FTL_DEFAULT_FORMS_8(X)

// How a step kernel's loads and stores use the caches (ftl_cache_for).
enum FtlCache : int { kCacheDefault, kCacheThrough, kCacheStream };

// Form ids, beside the class ids in a batch's runs and spans: the form with M
// points on each of G lanes, and all forms in one kernel.
constexpr int ftl_wide_id(int m, int g) { return 256 + 32 * m + g; }
constexpr int ftl_wide_m(int id) { return (id - 256) / 32; }
constexpr int ftl_wide_g(int id) { return (id - 256) % 32; }
#define FTL_WIDE_ALL 128

// The exact classes that run four or more waves per SIMD, the class of 2 and 3
// points, and the forms of the other point counts in launches that fill the
// chip, all in one kernel.
#define FTL_TILES_ALL 129
#define FTL_DEFAULT_CLASSES(X)                                                              \
  X(0, 4, 1, false) X(1, 8, 1, false) X(2, 16, 1, false) X(4, 8, 2, false) X(5, 16, 2, false) \
  X(7, 4, 4, false) X(8, 8, 4, false) X(9, 16, 4, false) X(10, 4, 1, true) X(15, 4, 2, false)
