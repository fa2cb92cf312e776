/* What fg_sampler_hip_create leaves in device memory, against a stand-in for
 * the HIP calls it makes: hipMalloc hands out host memory full of words that a
 * destroyed sampler could have left there, each tagged with the first epoch a
 * new sampler uses.  No such word may survive in a region whose words are
 * polled by tag (lists, greedy composites, speculative keys).
 *
 * With the argument "slice": what fg_hip_output_slice_create allocates for the
 * sampled output of 64 tokens, and that it does with less when hipMalloc
 * refuses larger blocks. */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "fg_sampler_hip.h"

#define MAX_ROWS 3u
/* Wave slots of a sampler of MAX_ROWS rows: (1,024 workgroups + rows) * 4. */
#define SLOTS ((1024u + MAX_ROWS) * 4u)
static const uint64_t stale = (0x2000ull | 1u) << 50 | 12345u;

static struct {
    uint64_t *at;
    size_t bytes;
} blocks[64];
static unsigned count;

static size_t largest = SIZE_MAX; /* block that hipMalloc grants */

int hipMalloc(void **out, size_t bytes)
{
    if (bytes > largest) return 2;
    if (count == 64u || !(*out = aligned_alloc(256, (bytes + 255u) & ~(size_t)255u))) return 2;
    for (size_t i = 0; i < bytes / 8u; i++) ((uint64_t *)*out)[i] = stale;
    blocks[count].at = *out;
    blocks[count++].bytes = bytes;
    return 0;
}
int hipMemset(void *at, int value, size_t bytes)
{
    memset(at, value, bytes);
    return 0;
}
int hipFree(void *at)
{
    free(at);
    return 0;
}
int hipGetDevice(int *device)
{
    *device = 0;
    return 0;
}
int hipDeviceGetAttribute(int *value, int attribute, int device)
{
    (void)attribute, (void)device;
    *value = 256;
    return 0;
}
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }

/* Bytes of the largest block of a whole-head slice for 64 tokens. */
static size_t slice_block(uint32_t vocab)
{
    fg_hip_output_slice *s = NULL;
    fg_error err;
    size_t most = 0;
    count = 0;
    if (fg_hip_output_slice_create(&s, vocab, 1u, 0u, vocab, 64u, &err) != FG_OK) return 0;
    for (unsigned b = 0; b < count; b++)
        if (blocks[b].bytes > most) most = blocks[b].bytes;
    fg_hip_output_slice_destroy(s);
    return most;
}

static int slice(void)
{
    static const size_t row = 248320u * 4u;
    const size_t all = slice_block(248320u), wide = slice_block(1000000u);
    largest = 20u * row;
    const size_t less = slice_block(248320u);
    largest = row - 1u;
    const size_t none = slice_block(248320u);
    printf("%zu %zu %zu %zu\n", all, wide, less, none);
    return all == 64u * row && wide && wide <= (64u << 20) && less == 16u * row && !none ? 0 : 1;
}

int main(int argc, char **argv)
{
    if (argc > 1) return strcmp(argv[1], "slice") ? 2 : slice();
    fg_sampler_hip *s = NULL;
    fg_error err;
    unsigned lists = 0, words = 0, bad = 0;
    if (fg_sampler_hip_create(&s, 5000u, MAX_ROWS, &err) != FG_OK) return 2;
    for (unsigned b = 0; b < count; b++) {
        const int list = blocks[b].bytes == (size_t)SLOTS * 64u * 8u;
        const int word = blocks[b].bytes == (size_t)SLOTS * 8u; /* greedy, speculative keys */
        lists += list, words += word;
        for (size_t i = 0; (list || word) && i < blocks[b].bytes / 8u; i++)
            if (blocks[b].at[i]) {
                printf("block %u of %zu bytes keeps a word of before\n", b, blocks[b].bytes);
                bad++;
                break;
            }
    }
    fg_sampler_hip_destroy(s);
    printf("%u lists, %u word regions, %u uncleared\n", lists, words, bad);
    return lists == 1u && words == 2u && !bad ? 0 : 1;
}
