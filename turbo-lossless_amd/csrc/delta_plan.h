// Which runs of the delta rule go sixteen tokens at a time (delta_rule.hip), and what their chunks take of the workspace (host and device).
#pragma once

namespace delta_rule {

constexpr int CHUNK = 16, CD = 64;                         // tokens of a chunk; key channels a head is padded to
constexpr int CHUNK_MAX_RANK = 512;                        // of the decay: what LDS has room for
// A chunk in the workspace: six arrays of 16 x 64 floats and the chunk's decay per key channel.
constexpr int CHUNK_FLOATS = 6 * CHUNK * CD + CD;
// Fewest tokens taken in chunks, whole calls, us, token by token against chunks: 16 heads of 64, 40 / 48 / 49 / 52 / 64 / 100 / 512 tokens 16.3 / 16.8 /
// 17.2 / 18.0 / 18.7 / 24.4 / 72.4 against 17.7 / 16.9 / 17.9 / 17.8 / 17.9 / 20.2 / 45.1 (a fourth chunk at 49); 24 heads of 48, 49 / 52 tokens 17.9 / 18.7
// against 18.4 / 18.3; 64 heads of 64, 52 / 512 22.3 / 105.4 against 21.6 / 73.0.
constexpr int CHUNK_FROM = 52;
// The most a chunk's floats come to per token of a run: 52 tokens are four chunks, 65 five.
constexpr int CHUNK_ROW = (CHUNK_FLOATS + 12) / 13;
static_assert(CHUNK_FROM == 52, "CHUNK_ROW is that of the shortest run of four chunks");

// The scan addresses its operands and its outputs by 32-bit offsets, in bytes from the head's first, and leaves it to the ends of the two
// buffers to drop what lies past the last token: three chunks are requested ahead.
constexpr int CHUNKS_PAST = 3;
inline bool chunk_offsets_fit(int heads, int dim, int n)
{
    const long long chunks = ((long long)n + CHUNK - 1) / CHUNK + CHUNKS_PAST, limit = 1ll << 31;
    return chunks * CHUNK * heads * dim * 4 < limit && chunks * CHUNK_FLOATS * 4 < limit;
}

// The factors of a chunk are those of decay rates up to one.  Heads of 16 channels: sums so short that token by token is the more exact,
// 1.37e-7 against 1.46e-7 over 48 tokens.
inline bool takes_chunks(int heads, int dim, int rank, int n, float decay_rate)
{
    return dim >= 32 && dim <= CD && rank <= CHUNK_MAX_RANK && n >= CHUNK_FROM && decay_rate >= 0.0f && decay_rate <= 1.0f && chunk_offsets_fit(heads, dim, n);
}

}  // namespace delta_rule
