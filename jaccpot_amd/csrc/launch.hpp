// Launch-side helpers shared by the .hip translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "common.hpp"

namespace jfm {

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

inline int32_t check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(JFM_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return JFM_OK;
}

// Consecutive levels of a tree sweep: offsets into the level-ordered node list,
// passed by value.
constexpr int kMaxSpan = 64;
struct LevelSpan {
  int32_t n;  // levels
  int32_t off[kMaxSpan + 1];
};

// Walks the levels of a sweep in order: `span(LevelSpan)` for runs of two or more
// consecutive levels of at most `small` nodes (at most kMaxSpan levels at a time),
// `level(first node, count)` for every other level.  Empty levels are skipped.
template <typename Span, typename Level>
inline void for_level_spans(const int32_t* off, int32_t nlev, int32_t small, Span span, Level level) {
  LevelSpan sp;
  sp.n = 0;
  auto flush = [&] {
    if (sp.n == 1) level(sp.off[0], sp.off[1] - sp.off[0]);
    if (sp.n > 1) span(sp);
    sp.n = 0;
  };
  for (int32_t l = 0; l < nlev; ++l) {
    const int32_t a = off[l], count = off[l + 1] - a;
    if (count <= 0) continue;
    if (count > small) {
      flush();
      level(a, count);
      continue;
    }
    if (sp.n == kMaxSpan) flush();
    if (sp.n == 0) sp.off[0] = a;
    sp.off[++sp.n] = a + count;
  }
  flush();
}

inline bool valid_levels(const int32_t* off, int32_t nlev) {
  if (nlev < 0 || (nlev > 0 && !off)) return false;
  for (int32_t l = 0; l < nlev; ++l)
    if (off[l + 1] < off[l] || off[l] < 0) return false;
  return true;
}

inline bool valid_dtype(int32_t d) { return d == JFM_F32 || d == JFM_F64; }

}  // namespace jfm

// Expands the body with a constexpr int P for every order compiled into the library.
#define JFM_FOR_ORDER(p, ...)                                                   \
  switch (p) {                                                                   \
    case 1: { constexpr int P = 1; __VA_ARGS__; } break;                                \
    case 2: { constexpr int P = 2; __VA_ARGS__; } break;                                \
    case 3: { constexpr int P = 3; __VA_ARGS__; } break;                                \
    case 4: { constexpr int P = 4; __VA_ARGS__; } break;                                \
    case 5: { constexpr int P = 5; __VA_ARGS__; } break;                                \
    case 6: { constexpr int P = 6; __VA_ARGS__; } break;                                \
    case 7: { constexpr int P = 7; __VA_ARGS__; } break;                                \
    case 8: { constexpr int P = 8; __VA_ARGS__; } break;                                \
    default:                                                                     \
      return ::jfm::fail(JFM_ERR_UNSUPPORTED, "order " + std::to_string(p) +     \
                                                  " is not compiled (1..8)");    \
  }

#define JFM_FOR_DTYPE(dtype, ...)                 \
  if ((dtype) == JFM_F32) {                        \
    using T = float;                               \
    __VA_ARGS__;                                   \
  } else if ((dtype) == JFM_F64) {                 \
    using T = double;                              \
    __VA_ARGS__;                                   \
  } else {                                         \
    return ::jfm::fail(JFM_ERR_ARG, "bad dtype");  \
  }
