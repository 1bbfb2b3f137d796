// Whether the shared expert's tiles of a matrix-core pass go along in the routed experts' launches (k_mfma_with_shared) or run
// on a stream beside the router, the routing and the dispatch tables.
#pragma once

#include <stddef.h>

namespace xabe {

// Token rows of a narrow tile, and the rows that one item of it covers of a gate (and up) matrix and of a down matrix.
constexpr int kNarrowRows = 64, kNarrowUpRows = 64, kNarrowDownRows = 128;

// An expert's share of the pass averages at most one block of 32 rows.
inline bool share_in_one_block(size_t tokens, size_t top_k, size_t num_experts) { return tokens * top_k <= 32 * num_experts; }

// Along, nothing is forked or joined (about 12 us, more where the host is what is waited for) and a persistent routed launch
// finds every CU free when it deals its items; but the shared expert's work no longer hides behind the launches in front.
// One layer, us, on a stream beside / along, uniform and skewed (`resident`: narrow workgroups that fit at once, 768):
//  - a share of more than 32 rows, where items are one block or two: 256 experts of 2048 x 512 (experts x hidden x width below),
//    1237 tokens 308 / 319 and 257 / 258;
//  - shared work of up to eight million weights made halfs, a few us at most: along.  4 x 2048 x 512, 64 tokens 83 / 53 and 85 / 56; 32 x 1024 x 512,
//    256 tokens 80 / 58 and 80 / 58, in buffers of 8192 86 / 77 and 88 / 76; 128 x 1024 x 512, 300: 104 / 102 and 85 / 73;
//  - fewer than two rounds of routed items: beside.  A shared item is then one more for a CU that had few, in down one more for a CU that had
//    one.  8 x 4096 x 14336, 64 tokens 452 / 500 and 460 / 516; 16 x 4096 x 6400, 64: 363 / 385 and 352 / 353; 32 x 4096 x 2048, 200: 250 / 260
//    and 248 / 249; 64 x 2048 x 1536, 100: 188 / 195 and 147 / 140; 8 x 8192 x 2048, 64: 208 / 225 and 209 / 228;
//  - from two rounds on: along.  256 x 2048 x 512, 64 tokens 206 / 201 and 97 / 92, 300: 247 / 246 and 148 / 137, 700: 262 / 258 and 189 / 182, 1024: 285 /
//    284 and 226 / 221; 512 x 2048 x 512, 512: 479 / 400 and 169 / 166; 256 x 7168 x 2048, 512: 2551 / 2425 and 2631 / 2359; 128 x 4096 x 1536, 200:
//    629 / 564 and 583 / 505; 128 x 2048 x 768, 256: 196 / 199 and 154 / 145 (two rounds exactly);
//  - unless the buffers are large for such a pass: the launches in front are as long as the buffers, and cover it all.  256 x 2048 x 512, 512
//    tokens in buffers of 3072: 266 / 264 and 176 / 170, 4096: 270 / 274 and 176 / 181, 8192: 294 / 301 and 200 / 207; 512 x 2048 x 512, 4096: 432 / 443 and
//    193 / 201; where a routed launch is long (from 3 * 2^28 weights a matrix stack) along all the same: 256 x 7168 x 2048, 8192: 2950 / 2703 and
//    2893 / 2631, 128 x 4096 x 1536, 200 tokens, 8192: 723 / 670 and 660 / 598.
inline bool shared_along(size_t tokens, size_t max_tokens, size_t top_k, size_t num_experts, size_t hidden, size_t intermediate, size_t resident) {
  if (!share_in_one_block(tokens, top_k, num_experts)) return false;
  const size_t matrix = hidden * intermediate, tiles = (tokens + kNarrowRows - 1) / kNarrowRows;
  if (tiles * 3 * matrix <= ((size_t)8 << 20)) return true;
  if (num_experts * (intermediate / kNarrowUpRows) < 2 * resident || num_experts * (hidden / kNarrowDownRows) < 2 * resident) return false;
  return max_tokens <= 3072 || num_experts * matrix >= ((size_t)3 << 28);
}

}  // namespace xabe
