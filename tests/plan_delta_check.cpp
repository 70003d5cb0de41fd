// Host program of tests/test_delta_plan.py: every run that takes_chunks() names has a workspace that holds its chunks and offsets, past
// its last token too, that 32 bits hold.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "delta_plan.h"

using namespace delta_rule;

static uint64_t state = 0x9e3779b97f4a7c15ull;
static uint32_t rnd()
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return (uint32_t)(state >> 11);
}

static int check(int heads, int dim, int n, bool* took)
{
    *took = takes_chunks(heads, dim, 64, n, 0.6f);
    if (!*took) return 0;
    const int64_t chunks = (n + CHUNK - 1) / CHUNK, step = (int64_t)heads * dim;
    if (chunks * CHUNK_FLOATS > (int64_t)n * CHUNK_ROW) return printf("%d tokens: %lld chunks past the workspace\n", n, (long long)chunks);
    // as delta_scan_kernel counts: the operands and outputs of the third chunk behind the one at work
    const int64_t ahead = chunks - 1 + 3, last_out = ahead * CHUNK * step + 15 * step + 15;
    if (last_out * 4 > INT32_MAX) return printf("%d heads of %d, %d tokens: output offset %lld\n", heads, dim, n, (long long)last_out * 4);
    if ((ahead + 1) * CHUNK_FLOATS * 4 > INT32_MAX) return printf("%d tokens: operand offset\n", n);
    return 0;
}

int main(int argc, char** argv)
{
    const long cases = argc > 1 ? atol(argv[1]) : 100000;
    long in = 0, out = 0;
    bool took;
    for (int n = 40; n < 5000; n++)
        if (check(1 + n % 64, 64, n, &took)) return 1;
    for (long i = 0; i < cases; i++) {
        const int heads = 1 + (int)(rnd() % 256), dim = 32 + (int)(rnd() % 33), n = 40 + (int)(rnd() % (1u << (6 + rnd() % 18)));
        if (check(heads, dim, n, &took)) return 1;
        (took ? in : out)++;
    }
    // what the rule names at the sizes of a model, and where it ends
    const struct { int heads, dim, n; bool chunks; } edges[] = {
        {16, 64, 51, false}, {16, 64, 52, true}, {16, 31, 512, false}, {16, 65, 512, false}, {64, 64, 100000, true}, {64, 64, 131072, false},
        {64, 64, 262145, false}, {16, 64, 1 << 20, false}, {1, 32, 1 << 20, true}, {1, 32, 1 << 21, false}};
    for (const auto& e : edges)
        if (takes_chunks(e.heads, e.dim, 64, e.n, 0.6f) != e.chunks) return printf("%d heads of %d, %d tokens: %d\n", e.heads, e.dim, e.n, !e.chunks);
    if (takes_chunks(16, 64, 64, 512, 1.01f) || takes_chunks(16, 64, 64, 512, -0.1f) || takes_chunks(16, 64, 64, 512, __builtin_nanf(""))) return printf("decay rates\n");
    if (!takes_chunks(16, 64, 512, 512, 0.6f) || takes_chunks(16, 64, 513, 512, 0.6f)) return printf("ranks\n");
    printf("ok: %ld in chunks, %ld not\n", in, out);
    return 0;
}
