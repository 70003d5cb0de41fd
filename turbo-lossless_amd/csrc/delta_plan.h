// Which runs of the delta rule go sixteen tokens at a time (delta_rule.hip), and what their chunks take of the workspace (host and device).
#pragma once

namespace delta_rule {

constexpr int CHUNK = 16, CD = 64;                         // tokens of a chunk; key channels a head is padded to
// A chunk in the workspace: six arrays of 16 x 64 floats and the chunk's decay per key channel.
constexpr int CHUNK_FLOATS = 6 * CHUNK * CD + CD;
// Fewest tokens taken in chunks, whole calls of 16 heads of 64, token by token against chunks: 31 / 33 tokens 15.4 / 15.9 us against 16.1 / 16.1,
// 64 / 100 / 512 tokens 19.4 / 24.5 / 72.6 against 15.8 / 18.3 / 37.7 (64 heads: 105.5 against 60.9).
constexpr int CHUNK_FROM = 40;
// The most a chunk's floats come to per token of a run: 49 tokens are four chunks.
constexpr int CHUNK_ROW = (4 * CHUNK_FLOATS + 48) / 49;
static_assert(CHUNK_FROM > 33 && CHUNK_FROM <= 49, "CHUNK_ROW is that of the shortest run of four chunks");

// The scan addresses its operands and its outputs by 32-bit offsets, in bytes from the head's first, and leaves it to the ends of the two
// buffers to drop what lies past the last token: up to three chunks gone through on zeros, and three requested ahead of those.
constexpr int CHUNKS_PAST = 6;
inline bool chunk_offsets_fit(int heads, int dim, int n)
{
    const long long chunks = ((long long)n + CHUNK - 1) / CHUNK + CHUNKS_PAST, limit = 1ll << 31;
    return chunks * CHUNK * heads * dim * 4 < limit && chunks * CHUNK_FLOATS * 4 < limit;
}

// The factors of a chunk are those of decay rates up to one.  Heads of 16 channels: sums so short that token by token is the more exact,
// 1.37e-7 against 1.46e-7 over 48 tokens.
inline bool takes_chunks(int heads, int dim, int n, float decay_rate)
{
    return dim >= 32 && dim <= CD && n >= CHUNK_FROM && decay_rate >= 0.0f && decay_rate <= 1.0f && chunk_offsets_fit(heads, dim, n);
}

}  // namespace delta_rule
