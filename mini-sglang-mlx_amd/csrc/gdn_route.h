// Which kernel takes a call of the gated delta rule with more than a token a request (host code).
#pragma once
#include <algorithm>
#include <cstdint>

namespace msgl {

enum class GdnRoute { kTokens, kShort, kChunks };  // gdn_state.hip; gdn_short.hip; gdn_chunk.hip, gdn_long.hip

// Whether chunks of 64 are faster than token by token.  Their time for up to 64 tokens per request
// does not depend on their number: 12.8 us for each round of workgroups (two per value head, one per
// compute unit), or 9.2 us and 0.9 us per request of 32 heads where all requests go in pairs of waves (four
// workgroups per value head, in one round).  The token kernel's grows with the mean length, by 0.315 us per token while the requests
// run side by side and by 0.095 us per token and request of 32 heads beyond.  Both fitted to 1, 4, 16 and 64
// requests of 8, 16, 32 and 64 tokens; they meet between 15 and 30 tokens.
inline bool gdn_chunks_before_tokens(int64_t tokens, int64_t batch, int64_t hv, int64_t cus) {
  const double units = (double)(batch * hv) / 32, mean = (double)tokens / (double)batch;
  const double rounds = (double)((batch * hv * 2 + cus - 1) / cus);
  const bool pairs = batch <= 64 && batch * hv * 4 <= cus;
  return (pairs ? 9.2 + 0.9 * units : 12.8 * rounds) < 3.0 + 0.5 * units + mean * std::max(0.315, 0.13 + 0.095 * units);
}

// `longest`: most tokens of a request, 0: not known.
//
// By the mean length and units of 32 heads, even launches, us, token by token / in chunks of 16 / in chunks of 64:
//     1 unit: 4 tokens 5.7 / 5.8 / 9.2, 16 8.3 / 6.0 / 9.2, 32 13.0 / 6.7 / 9.3, 64 23 / 8.9 / 9.2
//     4:      4 tokens 9.8 / 7.1 / 12.1, 16 17 / 7.2 / 12.1, 32 27 / 8.2 / 12.1, 64 46 / 10.5 / 12.4
//     8:      4 tokens 16 / 9.7 / 25, 16 28 / 10.6 / 25, 48 62 / 13.0 / 25, 256 - / 40 / 56
//     16:     4 tokens 20 / 15 / 50, 16 38 / 15.5 / 50, 64 112 / 25 / 51, 256 - / 73 / 107
// Up to three tokens the token kernel is as fast (1.00-1.28 beyond 16 units, 1.03-1.14 up to 1, where this goes for up to 8 tokens).
//
// Against token by token chunks of 16 are faster whatever the lengths (850 launches of 1-200 requests, 4-64 heads, even, ragged, of
// one request 8 to 256 times as long as the others: 0.5, worst 1.03).  Against chunks of 64 they are where no request is long: its
// chunks come one after the other, 1.4 us for 16 tokens against 2.8 for 64, while the chunks of 64 take 8 us and more
// for each round of workgroups.  667 such launches, their time in chunks of 16 by that in chunks of 64: all 0.74 (geometric mean, 0.27-1.83: one
// of 4000 tokens among 47 of 40 500 us and 293, 2000 among 31 of 8 250 and 152, 720 among 15 single tokens 95 and 64); the 440
// that the sums below send there 0.575 (worst 0.98), the others 1.22, so that all take 0.694, and the faster way of each 0.689.  Where
// the longest is not known, chunks of 64 take what they are faster for than token by token, as one long request would have it.
inline GdnRoute gdn_route(int64_t tokens, int64_t batch, int64_t hv, int64_t longest, int64_t cus) {
  const int64_t heads = batch * hv;
  const int64_t least = heads <= 32 ? 9 : heads <= 64 || heads > 512 ? 4 : 2, most = heads <= 512 ? 49 : std::min<int64_t>(128, 12 + 3 * heads / 32);
  if (tokens < least * batch) return GdnRoute::kTokens;
  if (tokens >= most * batch) return GdnRoute::kChunks;
  if (!gdn_chunks_before_tokens(tokens, batch, hv, cus)) return GdnRoute::kShort;
  if (longest <= 0) return GdnRoute::kChunks;
  const double rounds = (double)((2 * heads + cus - 1) / cus);
  const double chain = 6.0 + 1.4 * (double)((longest + 15) / 16);
  return chain <= std::max(9.2 + 2.8 * (double)((longest + 63) / 64), 8.0 * rounds) ? GdnRoute::kShort : GdnRoute::kChunks;
}

}  // namespace msgl
