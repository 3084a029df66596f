// Chunk-wise mixed-precision Adam step for MI355X (gfx950, wave64).
//
// Everything here is HBM-bandwidth bound: 28 bytes move per element per step
// (read fp16 grad + fp32 param/m/v, write fp32 param/m/v + fp16 param) for
// ~20 flops.  No matrix cores are involved.  What the kernels are organised
// around, all of it measured on MI355X:
//   * one pass over the data, in place; per lane one 16-byte access to each
//     fp32 array and one 8-byte access to the fp16 array, so that every wave
//     instruction covers a contiguous span of whole cache lines;
//   * one small tile (256 elements) per single-wave workgroup and a CAP on
//     resident workgroups (9 per CU, enforced by requesting 17 KiB of unused
//     dynamic LDS; 11 with the hint below): the pass touches four arrays for
//     reading and the same four for writing, and HBM efficiency drops when the set of in-flight cache
//     lines gets wide; a narrow, steadily advancing window per array gave
//     6.3 TB/s where the fully occupied machine gave 5.3 TB/s (a plain
//     1-read-1-write copy peaks at 6.3-6.4 TB/s on the same GPU);
//   * chunk descriptors travel in the kernel-argument segment (64 per launch),
//     so a wave's first data load depends on one scalar load, not two; evenly
//     spaced chunks need 12 words, preloaded into scalar registers;
//   * lists too long for the caches stream past them: non-temporal loads AND
//     stores, and 11 instead of 9 workgroups per CU, 6.6 TB/s where plain
//     accesses gave 6.25 (either hint alone gains nothing or loses 6 %).
//
// Arithmetic contract (ps_arith.h).  Operator arithmetic: bit-exact with the
// explicit-intrinsic body of the reference operator
// (patrickstar/ops/csrc/adam/cpu_adam.cpp:91-141): every a*b+c the reference
// writes as SIMD_FMA is one __builtin_fmaf; every other operation is an
// individually rounded IEEE binary32 op.  Torch arithmetic: one rounding step
// per torch kernel of FP16Adam.torch_adam_update
// (patrickstar/ops/fp16_cpu_adam.py:259-277), as torch's GPU kernels round.
// Everything must be compiled with -ffp-contract=off and with correctly rounded
// fp32 divide and sqrt (hipcc's default), denormals preserved.
//
// Layout of the sources: ps_config.h (tuning knobs), ps_arith.h (step constants
// and per-element arithmetic), ps_tile.h (vector accesses, one tile per wave),
// ps_kernels.h (the kernels), this file (host state, launches, streaming of
// host-resident chunks, the C ABI).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <unordered_map>
#include <vector>

#include "ps_adam.h"

#include "ps_config.h"
#include "ps_arith.h"
#include "ps_tile.h"
#include "ps_kernels.h"

namespace {

// ------------------------------------------------------------------ errors

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int hip_fail(hipError_t e, const char* what)
{
    return fail(-(int)e, "%s: %s", what, hipGetErrorString(e));
}

#define PS_HIP(call)                                      \
    do {                                                  \
        hipError_t e_ = (call);                           \
        if (e_ != hipSuccess) return hip_fail(e_, #call); \
    } while (0)

// ------------------------------------------------------- host scalar state
//
// One object per optimizer id: the float scalars the reference keeps in
// Adam_Optimizer (cpu_adam.h:177-197) and their update rules.

struct HostAdam {
    float alpha, beta1, beta2, eps, weight_decay;
    float beta1_t = 1.0f, beta2_t = 1.0f;
    size_t step = 0;
    bool adamw;
    double grad_clamp = -1.0;  // FP16Adam.gradient_clipping; <= 0: off
    int arith = PS_ARITH_OPERATOR;  // arithmetic for chunks updated in place in HBM

    // cpu_adam.h:143-162
    void advance(size_t s, float b1, float b2)
    {
        if (b1 != beta1 || b2 != beta2) {
            step = s;
            beta1 = b1;
            beta2 = b2;
            beta1_t = (float)std::pow((double)b1, (double)s);
            beta2_t = (float)std::pow((double)b2, (double)s);
            return;
        }
        step += 1;
        if (step != s) {
            beta1_t = (float)std::pow((double)beta1, (double)s);
            beta2_t = (float)std::pow((double)beta2, (double)s);
            step = s;
        } else {
            beta1_t = beta1_t * beta1;
            beta2_t = beta2_t * beta2;
        }
    }
    // cpu_adam.h:163-170 (the bias-correction scalars follow in finish_consts)
    void set(float lr, float epsilon, float wd)
    {
        alpha = lr;
        eps = epsilon;
        weight_decay = wd;
    }
};

std::mutex g_registry_mutex;
std::unordered_map<int, std::shared_ptr<HostAdam>> g_registry;

std::shared_ptr<HostAdam> find_opt(int id)
{
    std::lock_guard<std::mutex> lock(g_registry_mutex);
    auto it = g_registry.find(id);
    return it == g_registry.end() ? nullptr : it->second;
}

// ------------------------------------------------------------ launch helpers

// The runtime refuses a launch whose grid times block size reaches 2^32 threads in a dimension.  Kernels that take one
// tile per single-wave workgroup are checked against kMaxGridX before anything is queued (2^26 - 1 tiles: chunks and
// tensors of up to 17 G elements); kernels that loop over their tiles are simply capped (grid_1d).
constexpr size_t kMaxGridX = 0xFFFFFFFFull / 64;
static_assert(kBlock == 64 && kScanBlock == 64, "kMaxGridX is for 64-thread workgroups");

constexpr int kMaxGridY = 65535;

constexpr size_t kMaxCopyBlocks = 0xFFFFFFFFull / kCopyBlock;  // of the gradient copy (2^24 - 1 spans of 2048 elements)

unsigned grid_1d(size_t n_blocks, size_t block_threads)
{
    const size_t most = 0xFFFFFFFFull / block_threads;
    size_t g = n_blocks < most ? n_blocks : most;
    return (unsigned)(g ? g : 1);
}

// Validated view of a host array of chunk descriptors.
struct ChunkList {
    const ps_chunk* chunks;
    int n_chunks;
    size_t chunk_numel;
    const size_t* used;  // per chunk: elements in front of the zero padding; nullptr: every chunk is full
    size_t tile;         // elements per workgroup of the kernel that will run over the list

    size_t numel_of(int i) const { return used ? used[i] : chunk_numel; }
};

// All descriptors are checked here, before anything is enqueued or any host state advances.
int make_chunk_list(ChunkList& a, const ps_chunk* chunks, int n_chunks, size_t chunk_numel, const size_t* used_numel,
                    size_t tile, bool fp16_only = false, const char* what = "chunk")
{
    if (n_chunks < 0) return fail(PS_ERR_BAD_ARG, "n_chunks = %d is negative", n_chunks);
    if (chunks == nullptr && n_chunks > 0) return fail(PS_ERR_BAD_ARG, "chunks is NULL");
    for (int i = 0; i < n_chunks; ++i) {
        const ps_chunk& c = chunks[i];
        if (!c.param_fp16 || (!fp16_only && (!c.param_fp32 || !c.exp_avg || !c.exp_avg_sq)))
            return fail(PS_ERR_BAD_ARG, "%s %d has a NULL payload address", what, i);
        if (used_numel && used_numel[i] > chunk_numel)
            return fail(PS_ERR_BAD_ARG, "%s %d: used_numel = %zu is beyond chunk_numel = %zu", what, i, used_numel[i],
                        chunk_numel);
    }
    a.chunks = chunks;
    a.n_chunks = n_chunks;
    a.chunk_numel = chunk_numel;
    a.used = used_numel;
    a.tile = tile;
    if ((chunk_numel + tile - 1) / tile > kMaxGridX)
        return fail(PS_ERR_BAD_ARG, "chunk_numel = %zu is beyond the launch grid", chunk_numel);
    return 0;
}

// Calls launch(batch, grid, index of the batch's first chunk) for every group of up to kBatch chunks.  The grid is
// as wide as the longest chunk of the batch; workgroups beyond a shorter chunk's end leave at once.
template <typename F>
int for_each_batch(const ChunkList& a, F launch)
{
    for (int first = 0; first < a.n_chunks; first += kBatch) {
        int n = a.n_chunks - first < kBatch ? a.n_chunks - first : kBatch;
        ChunkBatch b;
        memset(&b, 0, sizeof(b));
        size_t tiles = 0;
        for (int i = 0; i < n; ++i) {
            b.c[i] = a.chunks[first + i];
            b.n[i] = a.numel_of(first + i);
            tiles = std::max(tiles, (b.n[i] + a.tile - 1) / a.tile);
        }
        if (tiles == 0) continue;
        launch(b, dim3((unsigned)tiles, (unsigned)n), first);
        PS_HIP(hipGetLastError());
    }
    return 0;
}

size_t elements(const ChunkList& a)
{
    size_t n = 0;
    for (int i = 0; i < a.n_chunks; ++i) n += a.numel_of(i);
    return n;
}

// ---- streaming past the caches
//
// A pass over a list uses nothing twice, but its loads and stores go through the L2 and the memory-side cache like any
// other: what a kernel has written waits there, is written back when something else needs the room or the kernel ends, and
// is in the way of the loads.  With the non-temporal hint on loads AND stores (and 11 workgroups per CU instead of 9) it
// leaves at once.  24 x 64 Mi elements 7211 -> 6848 us host-decided, a device-decided step with its probe 7713 -> 7266; 8 x 64 Mi
// 2374 -> 2234 and 2572 -> 2394; one 64 Mi chunk 295 -> 280 and 324 -> 304.  The hint on the loads alone makes the same steps 6 %
// slower, on the stores alone nothing.
//
// Steps over a list that stays in the memory-side cache from one step to the next (256 MiB) want it there; others, because forward and
// backward went over more than the cache holds, do not, and a call does not know which it is.  Without / with the hint, the same list
// again and again: host-decided 8 Mi elements 28.8 / 36.7 us, 16 Mi 65.7 / 69.7, 18 Mi 73.4 / 78.7, 20 Mi 90.8 / 88.1, 22 Mi 98.0 / 97.0, 24 Mi 108.2 /
// 105.9, 26 Mi 118.3 / 115.4; device-decided 16 Mi 72.9 / 77.0, 18 Mi 79.8 / 85.9, 20 Mi 99.5 / 94.8, 22 Mi 104.4 / 103.9, 24 Mi 114.4 / 113.2, 26 Mi
// 123.8 / 122.3; device-decided tensors with numbers of their own 17.5 Mi 80.1 / 87.0, 20 Mi 101.2 / 98.5, 23 Mi 115.7 / 111.6, 26 Mi 129.2 / 122.9 (runs
// of one side differ by 2 to 8 us here, by 0.4 below).  Three lists in turn: host-decided 4 Mi 16.1 / 20.2, 8 Mi 38.9 / 37.3, 16 Mi 78.4 / 71.6, 24 Mi 112.8 / 106.8;
// device-decided 8 Mi 40.7 / 39.9, 16 Mi 85.3 / 77.8, 20 Mi 104.9 / 95.8, 26 Mi 134.6 / 122.5; tensors 17.5 Mi 94.5 / 86.9, 23 Mi 125.1 / 111.1.
// Up to some 18 Mi elements a list that is in the cache loses 5 to 27 % by the hint, and plain accesses stay.  From 20 to 24 Mi on the hint loses in neither state, and from there to the lines, 28 Mi for every kind of step, plain
// accesses give up 1 to 5 % with the list in the cache and 5 to 11 % with it elsewhere: the lines are held by the tests of the routes, where
// a list of 27 Mi does not stream.
//
// A tensor of the operator comes with others, and its launch ends when its stores have left the L2.  Tensors of one length one after the other,
// without / with the hint, 600 MiB of them: 96 Ki elements 2.40 / 2.27 us, 128 Ki 2.56 / 2.35, 144 Ki 2.68 / 2.40, 192 Ki 2.93 / 2.57, 256 Ki 3.19 / 2.74, 576 Ki
// 4.77 / 3.55; eight of them, in the caches: the same within 0.03 up to 224 Ki, 256 Ki 2.34 / 2.27, 576 Ki 3.70 / 3.34; one of 2.25 Mi 13.0 / 11.5.  The loop of a program
// takes the host 3.7 us a call, which hides all of that below the line (256 Ki): modules of hidden size 384 and 448 with a line of 256 / 128 Ki
// 816 / 823 and 426 / 427 us (runs differ by 16 to 40); in a graph 516 / 465 and 320 / 283.
//
// The probe in front of an update reads what the update reads next: of a list it takes as much through the caches as the
// memory-side one holds, where a streaming update finds it, and the rest past them.  Whole steps, everything past the caches / the first 112 Mi
// elements through them: 31 Mi 148.5 / 142.9 us, 48 Mi 228 / 224, 80 Mi 373 / 358, 104 Mi 490 / 480, 136 Mi 642 / 627, 3 x 72 Mi 1018 / 1008, 8 x 64 Mi
// 2419 / 2402; 199 tensors of BERT-base with a rate per layer 502.6 / 479.  (96 Mi and 128 Mi: the same within 0.3 %.)  A skipped step reads no
// gradients again and pays for the slower probe: 48 Mi 62.6 / 64.3.  Of lists beyond 256 Mi it is 64 Mi.  Everything past the caches / 64 / 112 Mi: 8 x 64 Mi
// 2420.7 / 2411.5 / 2404.8 us, 5 x 56 Mi 1335.8 / 1328.5 / 1320.4, 12 x 64 Mi 3666.6 / 3661.1 / 3657.2; skipped 615.6 / 614.3 / 615.0, 339.5 / 341.3 / 341.3,
// 922.2 / 918.6 / 918.4, where runs differ by 3 to 10: 112 Mi there as well would give a clean step 0.1 to 0.6 % more at no cost that shows.
//
// A store that fills a 64-byte line in part only must not leave at once: lists whose phases differ by 16 or 32 bytes ran
// 5 to 6 % slower with the hint, by 64 6 % faster.
constexpr size_t kStreamElements = (size_t)28 << 20, kStreamElementsGated = (size_t)28 << 20, kScanKeepElements = (size_t)112 << 20,
                 kScanKeepOfLong = (size_t)256 << 20, kScanKeepLong = (size_t)64 << 20,
                 kFlatStreamElements = (size_t)256 << 10;
// How many tiles of the probe go through the caches.
uint32_t probe_keeps(const ChunkList& a) { return (uint32_t)((elements(a) > kScanKeepOfLong ? kScanKeepLong : kScanKeepElements) / kScanTile); }
bool whole_lines(const void* p32, const void* m32, const void* v32, const void* h16)
{
    return ((reinterpret_cast<uintptr_t>(p32) | reinterpret_cast<uintptr_t>(m32) | reinterpret_cast<uintptr_t>(v32) |
             reinterpret_cast<uintptr_t>(h16)) & 63u) == 0;
}
bool streams(const ChunkList& a, bool gated)
{
    if (elements(a) < (gated ? kStreamElementsGated : kStreamElements)) return false;
    for (int i = 0; i < a.n_chunks; ++i)
        if (!whole_lines(a.chunks[i].param_fp32, a.chunks[i].exp_avg, a.chunks[i].exp_avg_sq, a.chunks[i].param_fp16)) return false;
    return true;
}

// Dynamic LDS of a launch of the update, one tile a workgroup: the request that caps the resident workgroups per CU, except where
// all of the launch's workgroups fit the GPU at once (256 CUs with 32 waves each).  The cap keeps the window of lines in flight narrow
// while workgroups follow one another; a launch that has no second round only waits for its first one to end.  Capped / not, device
// time in a graph, host-decided step over one chunk of 768 Ki / 1 Mi / 1.25 Mi / 1.5 Mi / 2 Mi elements in the caches 4.3 / 3.9, 5.6 / 5.1, 6.3 / 5.6, 6.8 / 6.0,
// 8.0 / 6.9 us, in memory 6.6 / 6.0, 8.0 / 7.9, 9.5 / 9.4, 10.8 / 10.8, 13.5 / 13.8; device-decided, probe included, in the caches 7.1 / 6.5, 8.6 / 7.9, 9.4 / 8.4,
// 10.1 / 8.9, 11.9 / 10.3, in memory 8.9 / 8.3, 10.3 / 9.8, 11.9 / 11.6, 13.3 / 13.1, 16.1 / 16.4.  Tensors with numbers of their own 1.07 M elements 6.4 / 5.8, 2.1 M 10.2 /
// 8.5; one tensor of the operator 768 Ki 5.35 / 4.6, 1 Mi 6.35 / 6.15, 2 Mi 10.7 / 10.65, beyond the line 2.5 Mi 12.9 / 13.05.  Beyond it
// the cap pays: one chunk of 3 Mi in memory 18.6 / 19.3, 16 Mi 53.3 / 54.8, 26 Mi 116 / 130.  The line is that of lists in the caches: from 1.5 Mi elements
// (host-decided; device-decided 1.75 Mi) up to it a list in memory loses up to 2.5 %, where one in the caches gains 11 to 13 %.
constexpr size_t kResidentTiles = PS_RESIDENT_TILES;
unsigned capped_lds(dim3 grid, unsigned request) { return (size_t)grid.x * grid.y <= kResidentTiles ? 0 : request; }
template <bool NT>
unsigned capped_lds(dim3 grid)
{
    return capped_lds(grid, NT ? kStreamLdsBytes : kLdsBytes);
}

// launch(std::true_type or std::false_type): whether the kernel is the one with the non-temporal hint.
template <typename F>
void with_hint(bool nt, F launch)
{
    if (nt)
        launch(std::true_type{});
    else
        launch(std::false_type{});
}

// A list whose chunks follow one another at one distance, all of one length but perhaps the last (EvenChunk).
using EvenList = EvenBatch;

// Lists of up to this many elements take the kernels for it.  Longer ones are bound by memory from the first tile to the
// last: even / general kernels host-decided 558.1 / 559.2 us for 128 Mi elements, 2216 / 2217 for 512 Mi, 6719 / 6734 for 1.5 Gi;
// device-decided with the probe 1189.7 / 1193.6 for 256 Mi, 2368 / 2373 and 7154 / 7138.  (The lines are from plain accesses, where the
// general kernels were a little faster from there on: 7226 / 7236 and 7176 / 7209 for 1.5 Gi.)
constexpr size_t kMaxEvenElements = (size_t)96 << 20, kMaxEvenElementsGated = (size_t)256 << 20;
bool even_list(const ChunkList& a, size_t most, EvenList* out, bool fp16_only = false)
{
    const int n = a.n_chunks;
    if (n < 1 || n > kMaxGridY || a.numel_of(0) > most / n) return false;
    const size_t numel = a.numel_of(0), last = a.numel_of(n - 1);
    if (numel == 0 || numel > 0xFFFFFFFFu || last > numel) return false;
    auto addr = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
    const ps_chunk& f = a.chunks[0];
    const uintptr_t apart = n > 1 ? addr(a.chunks[1].param_fp16) - addr(f.param_fp16) : 0;  // bytes; a lower address: huge
    if (apart / 2 > 0xFFFFFFFFu || apart % 16 || addr(f.param_fp16) % 16) return false;
    if (!fp16_only && (addr(f.param_fp32) | addr(f.exp_avg) | addr(f.exp_avg_sq)) % 16) return false;
    for (int i = 1; i < n; ++i) {
        const ps_chunk& c = a.chunks[i];
        const uintptr_t d = apart * (uintptr_t)i;
        if (addr(c.param_fp16) - addr(f.param_fp16) != d || (i < n - 1 && a.numel_of(i) != numel)) return false;
        if (!fp16_only && (addr(c.param_fp32) - addr(f.param_fp32) != 2 * d || addr(c.exp_avg) - addr(f.exp_avg) != 2 * d ||
                           addr(c.exp_avg_sq) - addr(f.exp_avg_sq) != 2 * d))
            return false;
    }
    *out = EvenList{f, (uint32_t)(apart / 2), (uint32_t)numel, (uint32_t)(n - 1), (uint32_t)(numel - last)};
    return true;
}
dim3 even_grid(const EvenList& e, size_t tile) { return dim3((unsigned)((e.numel + tile - 1) / tile), e.last + 1); }

constexpr FirstCall kNoFirstCall{-1, 0, 0, 0, 0, 0, 0};

// Validated copy of a ps_call_pattern: how many operator calls the reference makes in the step and
// which elements its first call covers, as a chunk index over the call's whole list.
struct Calls {
    int64_t n_calls = 1;
    int64_t first_chunk = -1;  // -1: the first call's span is not needed (one call, or no elements)
    uint64_t lo = 0, hi = 0;

    // The span as the launch of chunks [batch_first, batch_first + n) sees it.
    FirstCall in_batch(int64_t batch_first, int n) const
    {
        FirstCall fc = kNoFirstCall;
        if (first_chunk >= batch_first && first_chunk < batch_first + n) {
            fc.chunk = (int)(first_chunk - batch_first);
            fc.lo = lo;
            fc.hi = hi;
            fc.lo_tile = (uint32_t)(lo / kTile);
            fc.hi_tile = (uint32_t)((hi + kTile - 1) / kTile);
            fc.in_lo = (uint32_t)((lo + kTile - 1) / kTile);
            fc.in_hi = (uint32_t)(hi / kTile);
        }
        return fc;
    }
};

int make_calls(Calls& out, const ps_call_pattern* calls, int64_t n_chunks_total, size_t chunk_numel)
{
    out = Calls();
    if (calls == nullptr) return 0;
    if (calls->n_calls < 1) return fail(PS_ERR_BAD_ARG, "calls->n_calls = %lld must be at least 1", (long long)calls->n_calls);
    out.n_calls = calls->n_calls;
    if (calls->n_calls == 1 || calls->first_numel == 0) return 0;  // one call, or a first call without elements
    if (calls->first_chunk < 0 || calls->first_chunk >= n_chunks_total)
        return fail(PS_ERR_BAD_ARG, "calls->first_chunk = %lld is outside the list of %lld chunks",
                    (long long)calls->first_chunk, (long long)n_chunks_total);
    if (calls->first_offset > chunk_numel || calls->first_numel > chunk_numel - calls->first_offset)
        return fail(PS_ERR_BAD_ARG, "the first call's tensor (offset %llu, %llu elements) does not fit a chunk of %zu",
                    (unsigned long long)calls->first_offset, (unsigned long long)calls->first_numel, chunk_numel);
    out.first_chunk = calls->first_chunk;
    out.lo = calls->first_offset;
    out.hi = calls->first_offset + calls->first_numel;
    return 0;
}

template <int ARITH, int WD>
void launch_adam_batch_wd(const ChunkBatch& b, dim3 grid, const StepConsts& c, const FirstCall& fc, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        dim3 block(kBlock);
        if (c.unscale == UNSCALE_MUL)
            hipLaunchKernelGGL((adam_chunks_kernel<ARITH, WD, UNSCALE_MUL, NT>), grid, block, capped_lds<NT>(grid), s, b, c, fc);
        else if (ARITH == PS_ARITH_OPERATOR && c.unscale == UNSCALE_DIV)  // the torch formula never divides
            hipLaunchKernelGGL((adam_chunks_kernel<ARITH, WD, UNSCALE_DIV, NT>), grid, block, capped_lds<NT>(grid), s, b, c, fc);
        else
            hipLaunchKernelGGL((adam_chunks_kernel<ARITH, WD, UNSCALE_NONE, NT>), grid, block, capped_lds<NT>(grid), s, b, c, fc);
    });
}

template <int ARITH>
void launch_adam_batch_arith(const ChunkBatch& b, dim3 grid, const StepConsts& c, const FirstCall& fc, bool nt, hipStream_t s)
{
    if (c.wd_mode == WD_DECOUPLED)
        launch_adam_batch_wd<ARITH, WD_DECOUPLED>(b, grid, c, fc, nt, s);
    else if (c.wd_mode == WD_L2)
        launch_adam_batch_wd<ARITH, WD_L2>(b, grid, c, fc, nt, s);
    else
        launch_adam_batch_wd<ARITH, WD_NONE>(b, grid, c, fc, nt, s);
}

#define PS_EVEN(e) (e).first.param_fp32, (e).first.exp_avg, (e).first.exp_avg_sq, (e).first.param_fp16, (e).stride, (e).numel, (e).last, (e).short_by

template <int ARITH, int WD>
void launch_even_wd(const EvenList& e, const StepConsts& c, const FirstCall& fc, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        const dim3 grid = even_grid(e, kTile), block(kBlock);
        if (c.unscale == UNSCALE_MUL)
            hipLaunchKernelGGL((adam_even_chunks_kernel<ARITH, WD, UNSCALE_MUL, NT>), grid, block, capped_lds<NT>(grid), s, PS_EVEN(e), c, fc);
        else if (ARITH == PS_ARITH_OPERATOR && c.unscale == UNSCALE_DIV)
            hipLaunchKernelGGL((adam_even_chunks_kernel<ARITH, WD, UNSCALE_DIV, NT>), grid, block, capped_lds<NT>(grid), s, PS_EVEN(e), c, fc);
        else
            hipLaunchKernelGGL((adam_even_chunks_kernel<ARITH, WD, UNSCALE_NONE, NT>), grid, block, capped_lds<NT>(grid), s, PS_EVEN(e), c, fc);
    });
}

template <int ARITH>
void launch_even_arith(const EvenList& e, const StepConsts& c, const FirstCall& fc, bool nt, hipStream_t s)
{
    if (c.wd_mode == WD_DECOUPLED)
        launch_even_wd<ARITH, WD_DECOUPLED>(e, c, fc, nt, s);
    else if (c.wd_mode == WD_L2)
        launch_even_wd<ARITH, WD_L2>(e, c, fc, nt, s);
    else
        launch_even_wd<ARITH, WD_NONE>(e, c, fc, nt, s);
}

template <int ARITH>
void launch_even_gated(const EvenList& e, size_t chunk_numel, const GatedArgs& ga, const FirstCall& fc,
                       const ps_step_state* d_state, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        const dim3 grid = even_grid(e, kTile), block(kBlock);
        const bool decay = ARITH == PS_ARITH_OPERATOR ? (float)ga.wd > 0.0f : ga.wd != 0.0;
        if (decay && ga.adamw)
            hipLaunchKernelGGL((adam_even_chunks_gated_kernel<ARITH, WD_DECOUPLED, NT>), grid, block, capped_lds<NT>(grid), s, PS_EVEN(e), d_state, chunk_numel, ga, fc);
        else if (decay)
            hipLaunchKernelGGL((adam_even_chunks_gated_kernel<ARITH, WD_L2, NT>), grid, block, capped_lds<NT>(grid), s, PS_EVEN(e), d_state, chunk_numel, ga, fc);
        else
            hipLaunchKernelGGL((adam_even_chunks_gated_kernel<ARITH, WD_NONE, NT>), grid, block, capped_lds<NT>(grid), s, PS_EVEN(e), d_state, chunk_numel, ga, fc);
    });
}

// The three forms of weight decay: launch(std::integral_constant<int, WD_...>).  The operator tests its float weight decay "> 0"
// (cpu_adam.cpp:42), the torch formula "!= 0".
template <int ARITH, typename F>
void with_decay(const GatedArgs& ga, F launch)
{
    const bool decay = ARITH == PS_ARITH_OPERATOR ? (float)ga.wd > 0.0f : ga.wd != 0.0;
    if (decay && ga.adamw)
        launch(std::integral_constant<int, WD_DECOUPLED>{});
    else if (decay)
        launch(std::integral_constant<int, WD_L2>{});
    else
        launch(std::integral_constant<int, WD_NONE>{});
}

template <bool NT>
dim3 with_first(dim3 grid)
{
    return dim3(grid.x + kInFront<NT>, grid.y);
}

template <int ARITH>
void launch_even_closing(const EvenList& e, size_t chunk_numel, const GatedArgs& ga, const FirstCall& fc, const Closing& cl, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        with_decay<ARITH>(ga, [&](auto wd) {
            constexpr bool NT = decltype(hint)::value;
            constexpr int WD = decltype(wd)::value;
            const dim3 grid = even_grid(e, kTile);
            hipLaunchKernelGGL((adam_even_chunks_closing_kernel<ARITH, WD, NT>), with_first<NT>(grid), dim3(kBlock), capped_lds<NT>(grid), s,
                               PS_EVEN(e), &cl.x->opened, chunk_numel, ga, fc, cl);
        });
    });
}

template <int ARITH>
void launch_closing_batch(const ChunkBatch& b, dim3 grid, size_t chunk_numel, const GatedArgs& ga, const FirstCall& fc, const Closing& cl, hipStream_t s)
{
    with_decay<ARITH>(ga, [&](auto wd) {
        hipLaunchKernelGGL((adam_chunks_closing_kernel<ARITH, decltype(wd)::value>), with_first<false>(grid), dim3(kBlock), capped_lds<false>(grid), s, &cl.x->opened, b,
                           chunk_numel, ga, fc, cl);
    });
}

// `c` must have been built for `arith` (finish_consts / torch_consts).  `fc`: which elements of the
// batch the step's first operator call covers; the torch formula has no such distinction.
void launch_adam_batch(int arith, const ChunkBatch& b, dim3 grid, const StepConsts& c, const FirstCall& fc, bool nt,
                       hipStream_t s)
{
    if (arith == PS_ARITH_TORCH)
        launch_adam_batch_arith<PS_ARITH_TORCH>(b, grid, c, kNoFirstCall, nt, s);
    else
        launch_adam_batch_arith<PS_ARITH_OPERATOR>(b, grid, c, fc, nt, s);
}

template <int ARITH>
void launch_gated_batch_arith(const ChunkBatch& b, dim3 grid, size_t chunk_numel,
                              const GatedArgs& ga, const FirstCall& fc, const ps_step_state* d_state,
                              bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        dim3 block(kBlock);
        // the operator tests its float weight decay "> 0" (cpu_adam.cpp:42), the torch formula "!= 0"
        const bool decay = ARITH == PS_ARITH_OPERATOR ? (float)ga.wd > 0.0f : ga.wd != 0.0;
        if (decay && ga.adamw)
            hipLaunchKernelGGL((adam_chunks_gated_kernel<ARITH, WD_DECOUPLED, NT>), grid, block, capped_lds<NT>(grid), s, b, chunk_numel, ga, fc, d_state);
        else if (decay)
            hipLaunchKernelGGL((adam_chunks_gated_kernel<ARITH, WD_L2, NT>), grid, block, capped_lds<NT>(grid), s, b, chunk_numel, ga, fc, d_state);
        else
            hipLaunchKernelGGL((adam_chunks_gated_kernel<ARITH, WD_NONE, NT>), grid, block, capped_lds<NT>(grid), s, b, chunk_numel, ga, fc, d_state);
    });
}

void launch_gated_batch(int arith, const ChunkBatch& b, dim3 grid, size_t chunk_numel,
                        const GatedArgs& ga, const FirstCall& fc, const ps_step_state* d_state,
                        bool nt, hipStream_t s)
{
    if (arith == PS_ARITH_TORCH)
        launch_gated_batch_arith<PS_ARITH_TORCH>(b, grid, chunk_numel, ga, kNoFirstCall, d_state, nt, s);
    else
        launch_gated_batch_arith<PS_ARITH_OPERATOR>(b, grid, chunk_numel, ga, fc, d_state, nt, s);
}

template <int ARITH, typename LIST>
void launch_small_step_arith(const LIST& b, const SmallStep& a, const GatedArgs& ga, const FirstCall& fc,
                             ps_step_state* d_state, StepScratch* scratch, hipStream_t s)
{
    dim3 grid(scratch ? (a.n_tiles + kSmallSpan - 1) / kSmallSpan : 1), block(kBlock, kSmallWaves);
    const bool decay = ARITH == PS_ARITH_OPERATOR ? (float)ga.wd > 0.0f : ga.wd != 0.0;
    if (decay && ga.adamw)
        hipLaunchKernelGGL((adam_small_step_kernel<LIST, ARITH, WD_DECOUPLED>), grid, block, 0, s, b, a, ga, fc, d_state, scratch);
    else if (decay)
        hipLaunchKernelGGL((adam_small_step_kernel<LIST, ARITH, WD_L2>), grid, block, 0, s, b, a, ga, fc, d_state, scratch);
    else
        hipLaunchKernelGGL((adam_small_step_kernel<LIST, ARITH, WD_NONE>), grid, block, 0, s, b, a, ga, fc, d_state, scratch);
}

template <typename LIST>
void launch_small_step(int arith, const LIST& b, const SmallStep& a, const GatedArgs& ga, const FirstCall& fc,
                       ps_step_state* d_state, StepScratch* scratch, hipStream_t s)
{
    if (arith == PS_ARITH_TORCH)
        launch_small_step_arith<PS_ARITH_TORCH>(b, a, ga, kNoFirstCall, d_state, scratch, s);
    else
        launch_small_step_arith<PS_ARITH_OPERATOR>(b, a, ga, fc, d_state, scratch, s);
}

template <typename LIST, bool NT>
unsigned list_lds(dim3 grid)
{
    if (std::is_same<LIST, NearBatch>::value) return capped_lds(grid, NT ? kStreamNearLdsBytes : kNearLdsBytes);
    return capped_lds<NT>(grid);
}

template <int ARITH, int WD, typename LIST>
void launch_tensors_wd(const LIST& b, dim3 grid, const StepConsts& c, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        dim3 block(kBlock);
        if (c.unscale == UNSCALE_MUL)
            hipLaunchKernelGGL((adam_tensors_kernel<LIST, ARITH, WD, UNSCALE_MUL, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, c);
        else if (ARITH == PS_ARITH_OPERATOR && c.unscale == UNSCALE_DIV)
            hipLaunchKernelGGL((adam_tensors_kernel<LIST, ARITH, WD, UNSCALE_DIV, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, c);
        else
            hipLaunchKernelGGL((adam_tensors_kernel<LIST, ARITH, WD, UNSCALE_NONE, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, c);
    });
}

template <int ARITH, typename LIST>
void launch_tensors_arith(const LIST& b, dim3 grid, const StepConsts& c, bool nt, hipStream_t s)
{
    if (c.wd_mode == WD_DECOUPLED)
        launch_tensors_wd<ARITH, WD_DECOUPLED>(b, grid, c, nt, s);
    else if (c.wd_mode == WD_L2)
        launch_tensors_wd<ARITH, WD_L2>(b, grid, c, nt, s);
    else
        launch_tensors_wd<ARITH, WD_NONE>(b, grid, c, nt, s);
}

template <int ARITH, typename LIST>
void launch_tensors_gated_arith(const LIST& b, dim3 grid, const GatedArgs& ga,
                                const ps_step_state* d_state, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        dim3 block(kBlock);
        const bool decay = ARITH == PS_ARITH_OPERATOR ? (float)ga.wd > 0.0f : ga.wd != 0.0;
        if (decay && ga.adamw)
            hipLaunchKernelGGL((adam_tensors_gated_kernel<LIST, ARITH, WD_DECOUPLED, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, ga, d_state);
        else if (decay)
            hipLaunchKernelGGL((adam_tensors_gated_kernel<LIST, ARITH, WD_L2, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, ga, d_state);
        else
            hipLaunchKernelGGL((adam_tensors_gated_kernel<LIST, ARITH, WD_NONE, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, ga, d_state);
    });
}

// The Python numbers of one step as they cross the boundary.
struct HyperParams {
    double lr, beta1, beta2, eps, wd;
    double loss_scale;  // <= 0: no loss scaler
    bool bias_correction;
    bool grad_f32 = false;  // the call's gradient tensor is binary32 (the clamp bound then narrows to float only)
};

// Host-decided step, operator arithmetic: narrow like the pybind signature of adam_update
// (float arguments, cpu_adam.cpp:700-712) and take the operator object through the n_calls
// adam_update calls of the reference's per-tensor loop, all with this step number: the first call's
// beta^t, then (from the second call on the object no longer moves) every later call's.
StepConsts operator_step_consts(HostAdam& o, size_t step, const HyperParams& hp, int64_t n_calls)
{
    o.advance(step, (float)hp.beta1, (float)hp.beta2);
    const float first_b1t = o.beta1_t, first_b2t = o.beta2_t;
    if (n_calls >= 2) o.advance(step, (float)hp.beta1, (float)hp.beta2);
    o.set((float)hp.lr, (float)hp.eps, (float)hp.wd);
    StepConsts c;
    finish_consts(c, o.alpha, o.beta1, o.beta2, o.eps, o.weight_decay, o.adamw, o.beta1_t,
                  o.beta2_t, hp.bias_correction, (float)hp.loss_scale, clamp_bound(o.grad_clamp, hp.loss_scale, hp.grad_f32));
    bias_scalars(o.alpha, first_b1t, first_b2t, hp.bias_correction, &c.first_step_size, &c.first_bc2inv);
    return c;
}

// Host-decided step, torch arithmetic (fp16_cpu_adam.py:412-413: Python's float ** int is the C
// library's pow).  The operator object is not touched: the reference does not call it here.
StepConsts torch_step_consts(const HostAdam& o, size_t step, const HyperParams& hp)
{
    double bc1 = 1.0, bc2 = 1.0;
    if (hp.bias_correction) {
        bc1 = 1.0 - std::pow(hp.beta1, (double)step);
        bc2 = 1.0 - std::pow(hp.beta2, (double)step);
    }
    StepConsts c;
    torch_consts(c, hp.lr, hp.beta1, hp.beta2, hp.eps, hp.wd, o.adamw, bc1, bc2, hp.loss_scale,
                 clamp_bound(o.grad_clamp, hp.loss_scale, hp.grad_f32));
    return c;
}

GatedArgs gated_args(const HostAdam& o, double lr, double eps, double wd, int bias_correction,
                     int64_t n_calls)
{
    GatedArgs ga;
    ga.lr = lr;
    ga.eps = eps;
    ga.wd = wd;
    ga.grad_clamp = o.grad_clamp;
    ga.n_calls = n_calls;
    ga.adamw = o.adamw ? 1 : 0;
    ga.bias_correction = bias_correction;
    return ga;
}

// ------------------------------------------- host-resident chunks: streaming
//
// Chunks that live in pinned host memory are updated in place when there are few of them (kMaxInPlaceChunks), else
// streamed through caller-owned staging buffers in HBM: H2D copies on one side stream, the fused kernel on a
// compute side stream, D2H copies on another side stream, tied together with
// events, so that with two or more staging slots the copy of chunk k+1 and the
// write-back of chunk k-1 overlap the kernel on chunk k.  Nothing blocks the
// host.  The streams and events are created once per device and kept.

constexpr int kMaxSlots = 8;

struct Pipeline {
    bool ready = false;
    std::mutex in_use;  // held by a call while it queues work on the side streams: calls on one device take turns
    hipStream_t h2d = nullptr, compute = nullptr, d2h = nullptr;
    hipEvent_t entry = nullptr;
    hipEvent_t joined[3] = {};  // one per side stream: "everything queued there so far"
    hipEvent_t h2d_done[kMaxSlots] = {}, compute_done[kMaxSlots] = {}, d2h_done[kMaxSlots] = {};
    bool slot_used[kMaxSlots] = {};

    int create()
    {
        // default priority on purpose
        PS_HIP(hipStreamCreateWithFlags(&h2d, hipStreamNonBlocking));
        PS_HIP(hipStreamCreateWithFlags(&compute, hipStreamNonBlocking));
        PS_HIP(hipStreamCreateWithFlags(&d2h, hipStreamNonBlocking));
        PS_HIP(hipEventCreateWithFlags(&entry, hipEventDisableTiming));
        for (hipEvent_t& e : joined) PS_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        for (int i = 0; i < kMaxSlots; ++i) {
            PS_HIP(hipEventCreateWithFlags(&h2d_done[i], hipEventDisableTiming));
            PS_HIP(hipEventCreateWithFlags(&compute_done[i], hipEventDisableTiming));
            PS_HIP(hipEventCreateWithFlags(&d2h_done[i], hipEventDisableTiming));
        }
        return 0;
    }

    // give back whatever a failed create() got as far as making
    void destroy()
    {
        for (hipStream_t* st : {&h2d, &compute, &d2h})
            if (*st) (void)hipStreamDestroy(*st), *st = nullptr;
        auto drop = [](hipEvent_t& e) {
            if (e) (void)hipEventDestroy(e), e = nullptr;
        };
        drop(entry);
        for (hipEvent_t& e : joined) drop(e);
        for (int i = 0; i < kMaxSlots; ++i) drop(h2d_done[i]), drop(compute_done[i]), drop(d2h_done[i]);
    }

    // A call begins: the copies and kernels it is about to queue on the side streams come after everything `caller`
    // has queued so far (gradients written, the device flag set) and after whatever an EARLIER call, possibly of
    // another host thread on another stream, left on any side stream (its staging slots may be the same memory).  For
    // one caller the second part is implied by the first (every call ends with join()).
    int begin(hipStream_t caller)
    {
        hipStream_t side[3] = {h2d, compute, d2h};
        for (int i = 0; i < 3; ++i) PS_HIP(hipEventRecord(joined[i], side[i]));
        PS_HIP(hipEventRecord(entry, caller));
        for (hipStream_t st : {h2d, compute}) {
            PS_HIP(hipStreamWaitEvent(st, entry, 0));
            for (int i = 0; i < 3; ++i)
                if (side[i] != st) PS_HIP(hipStreamWaitEvent(st, joined[i], 0));
        }
        for (int i = 0; i < kMaxSlots; ++i) slot_used[i] = false;
        return 0;
    }

    // Later work on `caller` comes after everything queued on the side streams so far.  Also used on
    // an error path, so that a half-queued step cannot race with whatever the caller does next.
    int join(hipStream_t caller)
    {
        hipStream_t side[3] = {h2d, compute, d2h};
        for (int i = 0; i < 3; ++i) {
            PS_HIP(hipEventRecord(joined[i], side[i]));
            PS_HIP(hipStreamWaitEvent(caller, joined[i], 0));
        }
        return 0;
    }
};

std::mutex g_pipeline_mutex;
std::unordered_map<int, Pipeline> g_pipelines;

int get_pipeline(Pipeline** out)
{
    int dev = 0;
    PS_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_pipeline_mutex);
    Pipeline* p = nullptr;
    try {
        p = &g_pipelines[dev];
    } catch (const std::exception&) {  // nothing may throw across the boundary
        return fail(PS_ERR_BAD_ARG, "no host memory for the streaming state of device %d", dev);
    }
    if (!p->ready) {
        if (int rc = p->create()) {
            p->destroy();
            return rc;
        }
        p->ready = true;
    }
    *out = p;
    return 0;
}

int check_slots(const ps_chunk* staging, int n_slots, bool need_state, bool need_fp16)
{
    if (n_slots < 1 || n_slots > kMaxSlots)
        return fail(PS_ERR_BAD_ARG, "n_slots = %d must be in 1..%d", n_slots, kMaxSlots);
    if (!staging) return fail(PS_ERR_BAD_ARG, "staging is NULL");
    for (int i = 0; i < n_slots; ++i) {
        if ((need_fp16 && !staging[i].param_fp16) ||
            (need_state && (!staging[i].param_fp32 || !staging[i].exp_avg || !staging[i].exp_avg_sq)))
            return fail(PS_ERR_BAD_ARG, "staging slot %d has a NULL buffer", i);
    }
    return 0;
}

// A host-resident chunk position may keep its fp16 payload in HBM (only the optimizer state lives in
// host memory): say for every position whether its fp16 address is device memory.
int fp16_payloads_in_hbm(const ps_chunk* host_chunks, int n, bool* in_hbm, bool* any_on_host)
{
    *any_on_host = false;
    for (int i = 0; i < n; ++i) {
        hipPointerAttribute_t attr;
        hipError_t e = hipPointerGetAttributes(&attr, host_chunks[i].param_fp16);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return fail(PS_ERR_BAD_ARG, "host chunk %d: the fp16 address is neither device nor pinned host memory (%s)",
                        i, hipGetErrorString(e));
        }
        in_hbm[i] = attr.type == hipMemoryTypeDevice;
        if (!in_hbm[i]) *any_on_host = true;
    }
    return 0;
}

// Few host chunks are updated where they are: the kernel reads and writes the pinned payloads over the link, both
// directions busy from the first tile to the last, where the copies leave one of them idle while the first chunk
// comes in and while the last one goes out.  In place moves 45.0 GB/s each way (whatever the launch shape: 1 to 4 tiles
// per workgroup, 2 to 32 workgroups per CU: 42.9 to 45.0) if the payloads start on KiB boundaries (from 64 bytes on 39,
// at any element 35), copies 57.1 one way and 48.3 each way when both are busy.  Chunks of 8 Mi elements, 12 B/element
// each way, copied / in place: one 3.73 / 2.47 ms, two 5.82 / 4.67, four 9.88 / 9.07, eight 18.11 / 17.90, nine 20.17 /
// 20.09, ten 22.21 / 22.28, twelve 26.34 / 26.69.
constexpr int kMaxInPlaceChunks = 8;

// Whether the update in place is no slower than the copies.  It shares the CUs with the resident chunks' kernels and is
// dispatched behind them, so the two take about as long as one after the other; copies run beside those kernels.  Two
// chunks of 8 Mi elements on the host, copied / in place: with 24 such chunks in HBM 5.81 / 5.22 ms, with 32 5.84 / 5.45,
// with 120 5.85 / 8.69; eight with 24 18.1 / 18.3.  At one element from a KiB boundary four chunks of 4 Mi 5.06 / 5.19 ms
// (at 4 elements), eight of 2 Mi 4.86 / 5.57.  Copies of small chunks are bound by their launches: 6267 elements 119 us
// for one, 172 for two, 416 for eight.
bool in_place_pays(const ChunkList& host, const bool* fp16_in_hbm, const ChunkList& resident)
{
    const double kUs = 1e-6, kGB = 1e9;
    double bytes = 0, longest = 0, resident_bytes = 0;  // of the host chunks: each way
    int n = 0;
    uintptr_t phase = 0;
    for (int i = 0; i < host.n_chunks; ++i) {
        if (host.numel_of(i) == 0) continue;
        const ps_chunk& c = host.chunks[i];
        const double b = (fp16_in_hbm[i] ? 12.0 : 14.0) * (double)host.numel_of(i);
        bytes += b;
        longest = std::max(longest, b);
        n += 1;
        phase |= (uintptr_t)c.param_fp32 | (uintptr_t)c.exp_avg | (uintptr_t)c.exp_avg_sq;
        if (!fp16_in_hbm[i]) phase |= (uintptr_t)c.param_fp16;
    }
    for (int i = 0; i < resident.n_chunks; ++i) resident_bytes += 28.0 * (double)resident.numel_of(i);
    const double link = bytes / ((phase & 1023) == 0 ? 45.0 * kGB : 35.0 * kGB);
    const double copies = std::max(60 * kUs + 40 * kUs * n, 2 * longest / (57.1 * kGB) + (bytes - longest) / (48.3 * kGB));
    return link + resident_bytes / (6200 * kGB) <= copies;
}

// Whether every payload of the list can be used by a kernel on the current device under the address the caller gave:
// pinned host memory of this device's making, mapped at its own address, or device memory.  (hipMemcpyAsync takes
// more than that: such payloads keep the copies.)
int mapped_in_place(const ps_chunk* host_chunks, int n, bool* out)
{
    int dev = 0;
    PS_HIP(hipGetDevice(&dev));
    *out = false;
    for (int i = 0; i < n; ++i) {
        const ps_chunk& c = host_chunks[i];
        for (const void* a : {(const void*)c.param_fp32, (const void*)c.exp_avg, (const void*)c.exp_avg_sq, (const void*)c.param_fp16}) {
            hipPointerAttribute_t attr;
            if (hipPointerGetAttributes(&attr, a) != hipSuccess) {
                (void)hipGetLastError();
                return 0;
            }
            if ((attr.type != hipMemoryTypeHost && attr.type != hipMemoryTypeDevice) || attr.device != dev || attr.devicePointer != a)
                return 0;
        }
    }
    *out = true;
    return 0;
}

}  // namespace

// ------------------------------------------- library-owned device scratch
//
// Partial results of ps_overflow_scan_chunks_noalloc: one word per workgroup of its first kernel.  A
// file-scope device array, so the entry point needs no allocation; every GPU the library runs on
// holds its own copy (4 MiB) at its own address until the process ends.  In host code the array's
// name is only a handle: the device address comes from hipGetSymbolAddress, once per device.
constexpr size_t kScratchWords = (size_t)1 << 20;
static __device__ __align__(256) uint32_t g_scan_scratch[kScratchWords];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
uint32_t* g_scratch_ptr[kMaxDevices] = {};

// The current device's copy of g_scan_scratch.
int scratch_address(uint32_t** out)
{
    int dev = 0;
    PS_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(PS_ERR_BAD_ARG, "device ordinal %d is beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        PS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(g_scan_scratch)));
        if (p == nullptr) return fail(PS_ERR_NO_DEVICE, "hipGetSymbolAddress gave no address for the scratch array");
        g_scratch_ptr[dev] = static_cast<uint32_t*>(p);
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

}  // namespace

// ====================================================================== ABI

extern "C" {

int ps_abi_version(void) { return PS_ABI_VERSION; }

const char* ps_last_error(void) { return g_err; }

int ps_adam_create(int optimizer_id, float alpha, float beta1, float beta2, float eps,
                   float weight_decay, int adamw_mode, int should_log)
{
    try {
        auto o = std::make_shared<HostAdam>();
        o->alpha = alpha;
        o->beta1 = beta1;
        o->beta2 = beta2;
        o->eps = eps;
        o->weight_decay = weight_decay;
        o->adamw = adamw_mode != 0;
        std::lock_guard<std::mutex> lock(g_registry_mutex);
        g_registry[optimizer_id] = o;
    } catch (const std::exception&) {  // nothing may throw across the boundary
        return fail(PS_ERR_BAD_ARG, "no host memory for optimizer %d", optimizer_id);
    }
    if (should_log) {
        printf("Adam Optimizer #%d is created with gfx950 HIP arithmetic capability.\n",
               optimizer_id);
        printf("Config: alpha=%f, betas=(%f, %f), weight_decay=%f, adam_w=%d\n", alpha, beta1,
               beta2, weight_decay, (int)(adamw_mode != 0));
    }
    return 0;
}

int ps_adam_set_grad_clamp(int optimizer_id, double gradient_clipping)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    o->grad_clamp = gradient_clipping;
    return 0;
}

int ps_adam_set_arithmetic(int optimizer_id, int arithmetic)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (arithmetic != PS_ARITH_OPERATOR && arithmetic != PS_ARITH_TORCH)
        return fail(PS_ERR_BAD_ARG, "arithmetic = %d is neither PS_ARITH_OPERATOR nor PS_ARITH_TORCH", arithmetic);
    o->arith = arithmetic;
    return 0;
}

int ps_adam_destroy(int optimizer_id)
{
    std::lock_guard<std::mutex> lock(g_registry_mutex);
    g_registry.erase(optimizer_id);
    return 0;
}

int ps_adam_update(int optimizer_id, size_t step, float lr, float beta1, float beta2, float epsilon,
                   float weight_decay, int bias_correction, float* d_params, const void* d_grads,
                   int grads_are_half, float* d_exp_avg, float* d_exp_avg_sq, size_t numel,
                   float loss_scale, uint16_t* d_param_fp16_out, ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (numel > 0 && (!d_params || !d_grads || !d_exp_avg || !d_exp_avg_sq))
        return fail(PS_ERR_BAD_ARG, "ps_adam_update: NULL tensor pointer");
    o->advance(step, beta1, beta2);
    o->set(lr, epsilon, weight_decay);
    if (numel == 0) return 0;
    StepConsts c;
    // the reference clamps gradients in Python before it calls the operator: not here
    finish_consts(c, o->alpha, o->beta1, o->beta2, o->eps, o->weight_decay, o->adamw, o->beta1_t,
                  o->beta2_t, bias_correction != 0, loss_scale, 0.0f);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t gsz = grads_are_half ? 2 : 4;
    const char* gbytes = static_cast<const char*>(d_grads);

    // element-wise pass over [lo, hi)
    auto scalar_span = [&](size_t lo, size_t hi) {
        if (hi <= lo) return;
        const size_t n = hi - lo;
        dim3 grid(grid_1d((n + kAuxBlock - 1) / kAuxBlock, kAuxBlock)), block(kAuxBlock);
        uint16_t* out = d_param_fp16_out ? d_param_fp16_out + lo : nullptr;
#define PS_FLAT(WD, HALF)                                                                      \
    hipLaunchKernelGGL((adam_flat_kernel<WD, HALF>), grid, block, 0, s, c, d_params + lo,      \
                       static_cast<const void*>(gbytes + lo * gsz), d_exp_avg + lo,            \
                       d_exp_avg_sq + lo, out, n)
        if (grads_are_half) {
            if (c.wd_mode == WD_DECOUPLED) PS_FLAT(WD_DECOUPLED, true);
            else if (c.wd_mode == WD_L2) PS_FLAT(WD_L2, true);
            else PS_FLAT(WD_NONE, true);
        } else {
            if (c.wd_mode == WD_DECOUPLED) PS_FLAT(WD_DECOUPLED, false);
            else if (c.wd_mode == WD_L2) PS_FLAT(WD_L2, false);
            else PS_FLAT(WD_NONE, false);
        }
#undef PS_FLAT
    };

    // Tensors handed to the operator are views at one element offset into the four chunk payloads, so their
    // addresses normally share a phase relative to 16-byte (4-element) boundaries: whole 256-element tiles with
    // vector accesses from the fp32 parameter's first 1 KiB boundary on (every wave access then covers one aligned
    // KiB); the up to 255 elements before it and the remainder behind the last whole tile go element-wise, in the
    // same launch.
    auto elem_phase = [](const void* a, size_t elem_size) -> int {
        uintptr_t u = reinterpret_cast<uintptr_t>(a);
        if (u % elem_size) return -1;
        return (int)((u / elem_size) & 3u);
    };
    // (momentum and variance may sit at any other element phase: the reference packs them in another order than the
    // parameters; their 16-byte accesses then go to 4-byte-aligned addresses)
    const int ph = elem_phase(d_params, 4);
    const bool vec_ok = ph >= 0 && numel >= 4096 && elem_phase(d_exp_avg, 4) >= 0 && elem_phase(d_exp_avg_sq, 4) >= 0 &&
                        elem_phase(d_grads, gsz) == ph &&
                        (d_param_fp16_out == nullptr || elem_phase(d_param_fp16_out, 2) == ph);
    const bool state_aligned = elem_phase(d_exp_avg, 4) == ph && elem_phase(d_exp_avg_sq, 4) == ph;
    if (!vec_ok) {
        scalar_span(0, numel);
        PS_HIP(hipGetLastError());
        return 0;
    }
    const size_t head = (size_t)((kTile - (reinterpret_cast<uintptr_t>(d_params) / sizeof(float)) % kTile) % kTile);
    // one tile per workgroup: a tensor beyond the launch grid (2^39 elements) goes in several launches
    const size_t max_tiles = kMaxGridX - 1;
    const bool nt = numel >= kFlatStreamElements && whole_lines(d_params + head, d_exp_avg + head, d_exp_avg_sq + head,
                                                                 d_param_fp16_out ? d_param_fp16_out + head : nullptr);
    size_t done = 0;  // elements behind the head that earlier launches of this call have covered
    const size_t body = numel - head;
    do {
        const size_t left = body - done;
        const bool last = left / kTile <= max_tiles;
        const size_t n_tiles = last ? left / kTile : max_tiles;
        const int tail = last ? (int)(left - n_tiles * kTile) : 0;
        const int this_head = done == 0 ? (int)head : 0;
        const size_t at = head + done;
        dim3 grid((unsigned)(n_tiles + (this_head + tail > 0 ? 1 : 0))), block(kBlock);  // + 1: the workgroup that does head and tail
        uint16_t* out = d_param_fp16_out ? d_param_fp16_out + at : nullptr;
#define PS_FLAT_VEC_5(WD, UNS, HALF, OUT, DWORD, NT)                                                                            \
    hipLaunchKernelGGL((adam_flat_vec_kernel<WD, UNS, HALF, OUT, DWORD, NT>), grid, block, capped_lds<NT>(grid), s, \
                       d_params + at, static_cast<const void*>(gbytes + at * gsz), d_exp_avg + at,                              \
                       d_exp_avg_sq + at, out, (uint32_t)n_tiles, this_head, tail, c)
#define PS_FLAT_VEC_4(WD, UNS, HALF, OUT)                    \
    do {                                                     \
        if (!state_aligned)                                  \
            PS_FLAT_VEC_5(WD, UNS, HALF, OUT, true, false);  \
        else if (nt)                                         \
            PS_FLAT_VEC_5(WD, UNS, HALF, OUT, false, true);  \
        else                                                 \
            PS_FLAT_VEC_5(WD, UNS, HALF, OUT, false, false); \
    } while (0)
#define PS_FLAT_VEC_3(WD, UNS, HALF)                       \
    do {                                                   \
        if (out != nullptr)                                \
            PS_FLAT_VEC_4(WD, UNS, HALF, true);            \
        else                                               \
            PS_FLAT_VEC_4(WD, UNS, HALF, false);           \
    } while (0)
#define PS_FLAT_VEC_2(WD, UNS)                             \
    do {                                                   \
        if (grads_are_half)                                \
            PS_FLAT_VEC_3(WD, UNS, true);                  \
        else                                               \
            PS_FLAT_VEC_3(WD, UNS, false);                 \
    } while (0)
#define PS_FLAT_VEC_1(WD)                                  \
    do {                                                   \
        if (c.unscale == UNSCALE_MUL)                      \
            PS_FLAT_VEC_2(WD, UNSCALE_MUL);                \
        else if (c.unscale == UNSCALE_DIV)                 \
            PS_FLAT_VEC_2(WD, UNSCALE_DIV);                \
        else                                               \
            PS_FLAT_VEC_2(WD, UNSCALE_NONE);               \
    } while (0)
        if (c.wd_mode == WD_DECOUPLED) PS_FLAT_VEC_1(WD_DECOUPLED);
        else if (c.wd_mode == WD_L2) PS_FLAT_VEC_1(WD_L2);
        else PS_FLAT_VEC_1(WD_NONE);
#undef PS_FLAT_VEC_1
#undef PS_FLAT_VEC_2
#undef PS_FLAT_VEC_3
#undef PS_FLAT_VEC_4
#undef PS_FLAT_VEC_5
        PS_HIP(hipGetLastError());
        done += n_tiles * kTile + tail;
    } while (done < body);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_adam_step_chunks(int optimizer_id, size_t step, double lr, double beta1, double beta2,
                        double epsilon, double weight_decay, int bias_correction,
                        const ps_chunk* chunks, int n_chunks, size_t chunk_numel,
                        const size_t* used_numel, const ps_call_pattern* calls, double loss_scale,
                        ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, used_numel, kTile)) return rc;
    Calls k;
    if (int rc = make_calls(k, calls, n_chunks, chunk_numel)) return rc;
    const HyperParams hp{lr, beta1, beta2, epsilon, weight_decay, loss_scale, bias_correction != 0};
    StepConsts c;
    if (o->arith == PS_ARITH_TORCH)
        c = torch_step_consts(*o, step, hp);
    else
        c = operator_step_consts(*o, step, hp, k.n_calls);
    if (!zeros_are_a_fixed_point(c)) a.used = nullptr;  // the padding is computed like everything else
    const int arith = o->arith;
    const bool nt = streams(a, false);
    hipStream_t s = static_cast<hipStream_t>(stream);
    EvenList e;
    if (even_list(a, kMaxEvenElements, &e)) {
        if (arith == PS_ARITH_TORCH)
            launch_even_arith<PS_ARITH_TORCH>(e, c, kNoFirstCall, nt, s);
        else
            launch_even_arith<PS_ARITH_OPERATOR>(e, c, k.in_batch(0, n_chunks), nt, s);
        PS_HIP(hipGetLastError());
        return 0;
    }
    return for_each_batch(a, [&](const ChunkBatch& b, dim3 grid, int first) {
        launch_adam_batch(arith, b, grid, c, k.in_batch(first, (int)grid.y), nt, s);
    });
}

int ps_adam_step_chunks_gated(int optimizer_id, double lr, double epsilon, double weight_decay,
                              int bias_correction, const ps_chunk* chunks, int n_chunks,
                              size_t chunk_numel, const size_t* used_numel,
                              const ps_call_pattern* calls, const ps_step_state* d_state,
                              ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, used_numel, kTile)) return rc;
    Calls k;
    if (int rc = make_calls(k, calls, n_chunks, chunk_numel)) return rc;
    const GatedArgs ga = gated_args(*o, lr, epsilon, weight_decay, bias_correction, k.n_calls);
    const int arith = o->arith;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool nt = streams(a, true);
    // (whether the padding may be left alone depends on the device-resident scalars: the kernel decides)
    EvenList e;
    if (even_list(a, kMaxEvenElementsGated, &e)) {
        if (arith == PS_ARITH_TORCH)
            launch_even_gated<PS_ARITH_TORCH>(e, chunk_numel, ga, kNoFirstCall, d_state, nt, s);
        else
            launch_even_gated<PS_ARITH_OPERATOR>(e, chunk_numel, ga, k.in_batch(0, n_chunks), d_state, nt, s);
        PS_HIP(hipGetLastError());
        return 0;
    }
    return for_each_batch(a, [&](const ChunkBatch& b, dim3 grid, int first) {
        launch_gated_batch(arith, b, grid, chunk_numel, ga, k.in_batch(first, (int)grid.y), d_state, nt, s);
    });
}

}  // extern "C"

namespace {

// ---------------------------------------------------------- tensor lists
//
// Where a tensor's tile grid starts (the fp32 parameter's first 1 KiB boundary; what lies in front of it is a tile of
// its own) and how many tiles it has.  Addresses that are not even element-aligned keep the plain numbering.
struct TensorItem {
    int index;  // in the caller's list
    uint32_t head;
    size_t body, tiles;
    int cls;  // the class of calls it belongs to (steps whose tensors carry their own numbers; 0 otherwise)
};
static_assert(kTile <= 256, "TensorBatch::lengths keeps the head length (up to kTile - 1 elements) in 8 bits");
static_assert(kMaxGridX * kTile <= kNumelMask, "TensorBatch::lengths keeps a length in 40 bits");

int check_tensor_list(const ps_chunk* tensors, const size_t* numels, int n_tensors)
{
    if (n_tensors < 0) return fail(PS_ERR_BAD_ARG, "n_tensors = %d is negative", n_tensors);
    if (n_tensors > 0 && (!tensors || !numels)) return fail(PS_ERR_BAD_ARG, "tensors or numels is NULL");
    for (int i = 0; i < n_tensors; ++i) {
        const ps_chunk& t = tensors[i];
        if (numels[i] > 0 && (!t.param_fp32 || !t.exp_avg || !t.exp_avg_sq || !t.param_fp16))
            return fail(PS_ERR_BAD_ARG, "tensor %d has a NULL address", i);
        if (numels[i] > kNumelMask || (numels[i] + kTile - 1) / kTile >= kMaxGridX)
            return fail(PS_ERR_BAD_ARG, "tensor %d: numel = %zu is beyond the launch grid", i, numels[i]);
    }
    return 0;
}

TensorItem tensor_item(const ps_chunk* tensors, const size_t* numels, int i, bool from_first_element = false)
{
    const uintptr_t p_addr = reinterpret_cast<uintptr_t>(tensors[i].param_fp32);
    size_t head = p_addr % sizeof(float) || from_first_element ? 0 : (kTile - (p_addr / sizeof(float)) % kTile) % kTile;
    if (head > numels[i]) head = numels[i];
    const size_t body = numels[i] - head;
    return TensorItem{i, (uint32_t)head, body, (head ? 1 : 0) + (body + kTile - 1) / kTile, 0};
}

// The same of tensors, whose tiles start at the parameter's KiB boundary.  Those with binary32 gradients (grad_f32(i)) never take
// the hint: they don't count.
template <typename F>
bool streams(const ps_chunk* tensors, const size_t* numels, int n_tensors, bool gated, F grad_f32)
{
    size_t total = 0;
    for (int i = 0; i < n_tensors; ++i)
        if (!grad_f32(i)) total += numels[i];
    if (total < (gated ? kStreamElementsGated : kStreamElements)) return false;
    for (int i = 0; i < n_tensors; ++i) {
        if (numels[i] < (size_t)kTile || grad_f32(i)) continue;
        const size_t head = tensor_item(tensors, numels, i).head;
        const ps_chunk& t = tensors[i];
        if (!whole_lines(t.param_fp32 + head, t.exp_avg + head, t.exp_avg_sq + head, t.param_fp16 + head)) return false;
    }
    return true;
}

// Calls launch(batch, grid, classes) for groups of the given tensors (all of them non-empty): longest first; one launch
// takes tensors of nearly the same length (its grid is as wide as the longest of them: at most a tenth of a
// launch's workgroups find nothing to do), short tensors all together.  `first_tensor`: the index (in the caller's
// list) of the tensor that is the step's first operator call, marked in its batch; -1: none.
//
// `classes`: which class each tensor of the batch belongs to.  max_classes == 0: the items' own class numbers.
// max_classes > 0: a launch takes at most that many distinct classes; its tensors' numbers are then 0, 1, ... in the
// order of their first tensor in the batch and classes.of[] says which of the items' classes each one is.
struct BatchClasses {
    int of[kNearBatch];
    int n;
};

// Number of a tensor's class in the launch that is being filled; -1: the launch holds as many classes as it may.
int class_in_batch(BatchClasses& bc, int cls, int max_classes)
{
    if (max_classes <= 0) return cls;
    for (int j = 0; j < bc.n; ++j)
        if (bc.of[j] == cls) return j;
    if (bc.n == max_classes) return -1;
    bc.of[bc.n] = cls;
    return bc.n++;
}

// Whether all of the items lie at the same place of their four lists (NearBatch): one distance from the fp32 parameter to
// momentum and to variance, and the fp16 slot half as far along as the parameter.  `lists`: where offset 0 lies.
bool near_lists(const std::vector<TensorItem>& items, const ps_chunk* tensors, ps_chunk* lists)
{
    const ps_chunk* low = nullptr;
    for (const TensorItem& it : items)
        if (!low || tensors[it.index].param_fp32 < low->param_fp32) low = &tensors[it.index];
    if (!low) return false;
    auto addr = [](const void* a) { return reinterpret_cast<uintptr_t>(a); };
    if ((addr(low->param_fp32) | addr(low->exp_avg) | addr(low->exp_avg_sq)) & 3u || addr(low->param_fp16) & 1u) return false;
    for (const TensorItem& it : items) {
        const ps_chunk& t = tensors[it.index];
        const uintptr_t d = addr(t.param_fp32) - addr(low->param_fp32);
        if (d & 3u || d / 4 + it.head > kNumelMask || it.body > 0xFFFFFFFFu) return false;
        if (addr(t.exp_avg) - addr(low->exp_avg) != d || addr(t.exp_avg_sq) - addr(low->exp_avg_sq) != d ||
            addr(t.param_fp16) - addr(low->param_fp16) != d / 2)
            return false;
    }
    *lists = *low;
    return true;
}

constexpr size_t kMaxNearElements = (size_t)256 << 20;  // of a list that takes NearBatch: see there

// The same for tensors of near_lists: a launch takes up to 208 of them, of up to 8 different lengths (within a tenth, and all
// of up to 32 tiles together: a workgroup that finds nothing to do costs 0.2 ns).
template <typename F>
int for_each_near_batch(const std::vector<TensorItem>& items, const ps_chunk* tensors, const ps_chunk& lists, int first_tensor,
                        int max_classes, F launch)
{
    constexpr size_t kShortTensorTiles = 32;
    NearBatch b;
    BatchClasses bc;
    size_t next = 0;
    while (next < items.size()) {
        memset(&b, 0, sizeof(b));
        memset(&bc, 0, sizeof(bc));
        b.lists = lists;
        b.first_call = -1;
        for (uint32_t& s : b.start) s = 0xFFFFFFFFu;
        size_t groups = 0;
        int in_batch = 0, segments = 0;
        for (; next < items.size() && in_batch < kNearBatch; ++in_batch, ++next) {
            const TensorItem& it = items[next];
            const uint32_t width = segments ? b.seg[segments - 1].width : 0;
            const bool opens = !segments || !(it.tiles * 10 >= (size_t)width * 9 || width <= kShortTensorTiles);
            const size_t wide = opens ? std::max<size_t>(it.tiles, 2) : width;
            if ((opens && segments == kSegments) || groups + wide > kMaxGridX) break;
            const int cls = class_in_batch(bc, it.cls, max_classes);
            if (cls < 0) break;
            if (opens) {
                const uint32_t magic = (uint32_t)((((uint64_t)1 << 32) + wide - 1) / wide);
                if (segments) b.start[segments - 1] = (uint32_t)groups;
                b.seg[segments++] = Segment{(uint32_t)groups, (uint32_t)in_batch, (uint32_t)wide, magic};
            }
            groups += wide;
            const uint64_t at = (uint64_t)(tensors[it.index].param_fp32 - lists.param_fp32) + it.head;
            b.at[in_batch] = at | ((uint64_t)cls << 40) | ((uint64_t)it.head << 56);
            b.numel[in_batch] = (uint32_t)it.body;
            if (it.index == first_tensor) b.first_call = in_batch;
        }
        launch(b, dim3((unsigned)groups), bc);
        PS_HIP(hipGetLastError());
    }
    return 0;
}

template <typename F>
int for_each_tensor_batch(std::vector<TensorItem>& items, const ps_chunk* tensors, int first_tensor, int max_classes,
                          F launch, bool grad_f32 = false)
{
    std::stable_sort(items.begin(), items.end(), [](const TensorItem& a, const TensorItem& b) { return a.tiles > b.tiles; });
    size_t elements = 0;
    for (const TensorItem& it : items) elements += it.head + it.body;
    ps_chunk lists;
    if (!grad_f32 && elements <= kMaxNearElements && near_lists(items, tensors, &lists))
        return for_each_near_batch(items, tensors, lists, first_tensor, max_classes, launch);
    constexpr size_t kShortTensorTiles = 256;
    TensorBatch b;
    BatchClasses bc;
    size_t next = 0;
    while (next < items.size()) {
        memset(&b, 0, sizeof(b));
        memset(&bc, 0, sizeof(bc));
        b.first_call = -1;
        const size_t widest = items[next].tiles;
        int in_batch = 0;
        while (next < items.size() && in_batch < kTensorBatch &&
               (items[next].tiles * 10 >= widest * 9 || widest <= kShortTensorTiles)) {
            const TensorItem& it = items[next];
            const int cls = class_in_batch(bc, it.cls, max_classes);
            if (cls < 0) break;  // the next launch starts with this tensor
            ps_chunk t = tensors[it.index];
            t.param_fp32 += it.head;
            t.exp_avg += it.head;
            t.exp_avg_sq += it.head;
            t.param_fp16 += it.head;
            b.t[in_batch] = t;
            b.lengths[in_batch] = (uint64_t)it.body | ((uint64_t)cls << 40) | ((uint64_t)it.head << 56);
            if (it.index == first_tensor) b.first_call = in_batch;
            in_batch += 1;
            next += 1;
        }
        launch(b, dim3((unsigned)widest, (unsigned)in_batch), bc);
        PS_HIP(hipGetLastError());
    }
    return 0;
}

// Weight-decay form of a call, as the two arithmetics decide it: the operator tests its float weight decay "> 0"
// (cpu_adam.cpp:42), the torch formula the Python number "!= 0".
int wd_mode_of(int arith, double wd, bool adamw)
{
    const bool decay = arith == PS_ARITH_OPERATOR ? (float)wd > 0.0f : wd != 0.0;
    return decay ? (adamw ? WD_DECOUPLED : WD_L2) : WD_NONE;
}

// `closing`: of a step whose launches read the copy of the state (NearBatch only); nullptr: they read the state.
template <int ARITH, int WD, typename LIST>
void launch_tensors_planned_wd(const LIST& b, dim3 grid, bool grad_f32,
                               const PlannedConsts* d_consts, const ps_step_state* d_state, const Closing* closing, bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        dim3 block(kBlock);
        if constexpr (std::is_same<LIST, TensorBatch>::value) {
            if (grad_f32) {
                hipLaunchKernelGGL((adam_tensors_planned_f32grad_kernel<ARITH, WD>), grid, block, capped_lds<false>(grid), s, b, d_consts, d_state);
                return;
            }
        }
        if constexpr (std::is_same<LIST, NearBatch>::value) {
            if (closing) {
                hipLaunchKernelGGL((adam_tensors_planned_closing_kernel<ARITH, WD, NT>), with_first<NT>(grid), block, (list_lds<LIST, NT>(grid)), s,
                                   b, d_consts, &closing->x->opened, *closing);
                return;
            }
        }
        hipLaunchKernelGGL((adam_tensors_planned_kernel<LIST, ARITH, WD, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, d_consts, d_state);
    });
}

template <int ARITH, typename LIST>
void launch_tensors_planned_arith(const LIST& b, dim3 grid, int wd_mode, bool grad_f32,
                                  const PlannedConsts* d_consts, const ps_step_state* d_state, const Closing* closing, bool nt, hipStream_t s)
{
    if (wd_mode == WD_DECOUPLED)
        launch_tensors_planned_wd<ARITH, WD_DECOUPLED>(b, grid, grad_f32, d_consts, d_state, closing, nt, s);
    else if (wd_mode == WD_L2)
        launch_tensors_planned_wd<ARITH, WD_L2>(b, grid, grad_f32, d_consts, d_state, closing, nt, s);
    else
        launch_tensors_planned_wd<ARITH, WD_NONE>(b, grid, grad_f32, d_consts, d_state, closing, nt, s);
}

// Numbers the distinct records (classes of calls) of a step by their bytes; records are zero-filled before they are
// set, so equal records have equal bytes.  Consecutive tensors mostly repeat the previous record.
template <typename T>
struct ClassTable {
    std::vector<T> records;
    std::vector<int> arith;
    std::unordered_map<std::string, int> by_bytes;
    int last = -1;

    int intern(const T& r, int a)
    {
        if (last >= 0 && arith[last] == a && memcmp(&records[last], &r, sizeof(T)) == 0) return last;
        std::string key(reinterpret_cast<const char*>(&r), sizeof(T));
        key.push_back((char)a);
        auto found = by_bytes.find(key);
        if (found == by_bytes.end()) {
            found = by_bytes.emplace(std::move(key), (int)records.size()).first;
            records.push_back(r);
            arith.push_back(a);
        }
        return last = found->second;
    }
    int size() const { return (int)records.size(); }
};

// What a launch of the per-tensor-numbers step is compiled for; classes that agree in it share launches.
struct Flavour {
    int arith, wd_mode, unscale;
    bool grad_f32;  // PS_TENSOR_GRAD_F32 tensors: binary32 gradients, no fp16 copy
    bool operator==(const Flavour& o) const
    {
        return arith == o.arith && wd_mode == o.wd_mode && unscale == o.unscale && grad_f32 == o.grad_f32;
    }
};

// What ClassTable keeps beside a record: the arithmetic, and whether the tensors' gradients are binary32.
int class_key(int arith, bool grad_f32) { return arith | (grad_f32 ? 2 : 0); }
int key_arith(int key) { return key & 1; }
bool key_grad_f32(int key) { return (key & 2) != 0; }
static_assert(PS_ARITH_OPERATOR == 0 && PS_ARITH_TORCH == 1, "class_key keeps the arithmetic in one bit");

template <int ARITH, int WD, int UNS, typename LIST>
void launch_tensors_each_uns(const LIST& b, dim3 grid, const ConstsBatch& cb, bool grad_f32,
                             bool nt, hipStream_t s)
{
    with_hint(nt, [&](auto hint) {
        constexpr bool NT = decltype(hint)::value;
        dim3 block(kBlock);
        if constexpr (std::is_same<LIST, TensorBatch>::value) {
            if (grad_f32) {
                hipLaunchKernelGGL((adam_tensors_each_f32grad_kernel<ARITH, WD, UNS>), grid, block, capped_lds<false>(grid), s, b, cb);
                return;
            }
        }
        hipLaunchKernelGGL((adam_tensors_each_kernel<LIST, ARITH, WD, UNS, NT>), grid, block, (list_lds<LIST, NT>(grid)), s, b, cb);
    });
}

template <int ARITH, int WD, typename LIST>
void launch_tensors_each_wd(const LIST& b, dim3 grid, const ConstsBatch& cb,
                            const Flavour& f, bool nt, hipStream_t s)
{
    if (f.unscale == UNSCALE_MUL)
        launch_tensors_each_uns<ARITH, WD, UNSCALE_MUL>(b, grid, cb, f.grad_f32, nt, s);
    else if (ARITH == PS_ARITH_OPERATOR && f.unscale == UNSCALE_DIV)  // the torch formula never divides
        launch_tensors_each_uns<ARITH, WD, UNSCALE_DIV>(b, grid, cb, f.grad_f32, nt, s);
    else
        launch_tensors_each_uns<ARITH, WD, UNSCALE_NONE>(b, grid, cb, f.grad_f32, nt, s);
}

template <int ARITH, typename LIST>
void launch_tensors_each_arith(const LIST& b, dim3 grid, const ConstsBatch& cb,
                               const Flavour& f, bool nt, hipStream_t s)
{
    if (f.wd_mode == WD_DECOUPLED)
        launch_tensors_each_wd<ARITH, WD_DECOUPLED>(b, grid, cb, f, nt, s);
    else if (f.wd_mode == WD_L2)
        launch_tensors_each_wd<ARITH, WD_L2>(b, grid, cb, f, nt, s);
    else
        launch_tensors_each_wd<ARITH, WD_NONE>(b, grid, cb, f, nt, s);
}

}  // namespace

extern "C" {

int ps_adam_step_tensors(int optimizer_id, size_t step, double lr, double beta1, double beta2,
                         double epsilon, double weight_decay, int bias_correction,
                         const ps_chunk* tensors, const size_t* numels, int n_tensors,
                         const ps_call_pattern* calls, double loss_scale, const ps_step_state* d_state,
                         ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (int rc = check_tensor_list(tensors, numels, n_tensors)) return rc;
    const int arith = o->arith;
    // One operator call per tensor.  Without a pattern the list is the whole step and tensors[0] its first call;
    // a pattern says how many calls the step has in all and which tensor of THIS list, if any, is the first.
    int64_t n_calls = n_tensors;
    int first_tensor = 0;
    if (calls != nullptr) {
        if (calls->n_calls < 1)
            return fail(PS_ERR_BAD_ARG, "calls->n_calls = %lld must be at least 1", (long long)calls->n_calls);
        n_calls = calls->n_calls;
        first_tensor = -1;
        if (calls->first_numel != 0) {
            if (calls->first_chunk < 0 || calls->first_chunk >= n_tensors)
                return fail(PS_ERR_BAD_ARG, "calls->first_chunk = %lld is outside the list of %d tensors",
                            (long long)calls->first_chunk, n_tensors);
            if (calls->first_offset != 0 || calls->first_numel != numels[calls->first_chunk])
                return fail(PS_ERR_BAD_ARG, "the first call is a whole tensor: calls->first_offset must be 0 and "
                            "calls->first_numel the length of tensor %lld", (long long)calls->first_chunk);
            first_tensor = (int)calls->first_chunk;
        }
    }
    if (arith != PS_ARITH_OPERATOR) first_tensor = -1;  // the torch formula has no first call
    StepConsts c;
    GatedArgs ga = gated_args(*o, lr, epsilon, weight_decay, bias_correction, n_calls);
    if (d_state == nullptr && n_tensors > 0) {
        const HyperParams hp{lr, beta1, beta2, epsilon, weight_decay, loss_scale, bias_correction != 0};
        c = arith == PS_ARITH_TORCH ? torch_step_consts(*o, step, hp) : operator_step_consts(*o, step, hp, n_calls);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    std::vector<TensorItem> items;
    try {
        items.reserve((size_t)n_tensors);
    } catch (const std::exception&) {  // nothing may throw across the boundary
        return fail(PS_ERR_BAD_ARG, "no host memory for a list of %d tensors", n_tensors);
    }
    for (int i = 0; i < n_tensors; ++i)
        if (numels[i] != 0) items.push_back(tensor_item(tensors, numels, i));
    const bool nt = streams(tensors, numels, n_tensors, d_state != nullptr, [](int) { return false; });
    return for_each_tensor_batch(items, tensors, first_tensor, 0, [&](const auto& b, dim3 grid, const BatchClasses&) {
        if (d_state == nullptr) {
            if (arith == PS_ARITH_TORCH)
                launch_tensors_arith<PS_ARITH_TORCH>(b, grid, c, nt, s);
            else
                launch_tensors_arith<PS_ARITH_OPERATOR>(b, grid, c, nt, s);
        } else {
            if (arith == PS_ARITH_TORCH)
                launch_tensors_gated_arith<PS_ARITH_TORCH>(b, grid, ga, d_state, nt, s);
            else
                launch_tensors_gated_arith<PS_ARITH_OPERATOR>(b, grid, ga, d_state, nt, s);
        }
    });
}

size_t ps_tensors_each_workspace_bytes(int n_tensors)
{
    return n_tensors > 0 ? (size_t)n_tensors * sizeof(PlannedConsts) : 0;
}

namespace {

int check_scratch(const void* d_scratch, size_t bytes)
{
    if (d_scratch != nullptr && (bytes < sizeof(StepScratch) || reinterpret_cast<uintptr_t>(d_scratch) % 64))
        return fail(PS_ERR_BAD_ARG, "d_scratch holds %zu bytes at %p; it needs %zu, 64-byte aligned", bytes, d_scratch, sizeof(StepScratch));
    return 0;
}

// The rest of a device-decided step with per-tensor numbers: the lists it probes, the scratch beside its state, and what its
// scale update is told.
struct WholeStep {
    const ChunkList& probed;
    StepScratch* scratch;
    ps_scale_record* log;
    int64_t log_capacity, operator_calls;
};

// Whether such lists can be done in one launch and those of the update.
bool lists_open_with_plan(const ChunkList& a, const ps_chunk* tensors, const size_t* numels, int n_tensors)
{
    if (a.n_chunks < 1 || a.n_chunks > kBatch) return false;
    size_t longest = 0, elements = 0;
    for (int i = 0; i < a.n_chunks; ++i) longest = std::max(longest, a.numel_of(i));
    if (longest == 0 || longest > 0xFFFFFFFFu) return false;
    std::vector<TensorItem> items;
    for (int i = 0; i < n_tensors; ++i) {
        if (numels[i] == 0) continue;
        items.push_back(tensor_item(tensors, numels, i));
        elements += numels[i];
    }
    ps_chunk lists;
    return elements <= kMaxNearElements && near_lists(items, tensors, &lists);  // (no item: false)
}

// Whether it is done in one launch and those of the update, the first of which replaces the state.
bool opens_with_plan(const WholeStep& w, int n_classes, const std::vector<int>& class_keys, const ps_chunk* tensors, const size_t* numels, int n_tensors)
{
    if (!w.scratch || n_classes > kOpenClasses) return false;
    for (int key : class_keys)
        if (key_grad_f32(key)) return false;
    return lists_open_with_plan(w.probed, tensors, numels, n_tensors);
}

int step_tensors_each(int optimizer_id, int bias_correction, const ps_chunk* tensors,
                      const size_t* numels, const ps_tensor_call* each, int n_tensors,
                      double loss_scale, ps_step_state* d_state, void* d_workspace,
                      size_t workspace_bytes, const WholeStep* whole, ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (int rc = check_tensor_list(tensors, numels, n_tensors)) return rc;
    if (n_tensors > 0 && !each) return fail(PS_ERR_BAD_ARG, "each is NULL");
    for (int i = 0; i < n_tensors; ++i) {
        const int a = each[i].arithmetic;
        if (a != -1 && a != PS_ARITH_OPERATOR && a != PS_ARITH_TORCH)
            return fail(PS_ERR_BAD_ARG, "each[%d].arithmetic = %d", i, a);
        if (d_state == nullptr && each[i].step < 1)
            return fail(PS_ERR_BAD_ARG, "each[%d].step = %lld: a host-decided step number is at least 1", i,
                        (long long)each[i].step);
        if (each[i].flags & ~PS_TENSOR_GRAD_F32) return fail(PS_ERR_BAD_ARG, "each[%d].flags = %d", i, each[i].flags);
    }
    if (d_state != nullptr && n_tensors > 0) {
        if (!d_workspace || workspace_bytes < ps_tensors_each_workspace_bytes(n_tensors))
            return fail(PS_ERR_BAD_ARG, "d_workspace holds %zu bytes; a device-decided step over %d tensors needs %zu",
                        d_workspace ? workspace_bytes : (size_t)0, n_tensors, ps_tensors_each_workspace_bytes(n_tensors));
        if (reinterpret_cast<uintptr_t>(d_workspace) % 16)
            return fail(PS_ERR_BAD_ARG, "d_workspace must be 16-byte aligned");
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool bias = bias_correction != 0;
    auto arith_of = [&](int i) { return each[i].arithmetic < 0 ? o->arith : each[i].arithmetic; };
    auto grad_f32_of = [&](int i) { return (each[i].flags & PS_TENSOR_GRAD_F32) != 0; };
    const bool nt = streams(tensors, numels, n_tensors, d_state != nullptr, grad_f32_of);
    try {
        // Calls that come out with the same constants form a class; class_of[i] says which one tensor i belongs to.
        std::vector<int> class_of((size_t)n_tensors, -1);
        if (d_state == nullptr) {
            // ---- host-decided: the operator object goes through the calls, in order
            ClassTable<StepConsts> classes;
            for (int i = 0; i < n_tensors; ++i) {
                const ps_tensor_call& e = each[i];
                const int arith = arith_of(i);
                const HyperParams hp{e.lr, e.beta1, e.beta2, e.eps, e.weight_decay, loss_scale, bias, grad_f32_of(i)};
                StepConsts c;
                memset(&c, 0, sizeof(c));
                if (arith == PS_ARITH_TORCH)
                    c = torch_step_consts(*o, (size_t)e.step, hp);
                else
                    c = operator_step_consts(*o, (size_t)e.step, hp, 1);
                class_of[i] = classes.intern(c, class_key(arith, grad_f32_of(i)));
            }
            const std::vector<StepConsts>& consts = classes.records;
            // one pass of launches per flavour (what the kernels are compiled for); inside it, tensors of any class
            std::vector<Flavour> flavours;
            std::vector<int> flavour_of(consts.size());
            for (size_t k = 0; k < consts.size(); ++k) {
                const Flavour f{key_arith(classes.arith[k]), consts[k].wd_mode, consts[k].unscale, key_grad_f32(classes.arith[k])};
                size_t j = 0;
                while (j < flavours.size() && !(flavours[j] == f)) ++j;
                if (j == flavours.size()) flavours.push_back(f);
                flavour_of[k] = (int)j;
            }
            std::vector<TensorItem> items;
            for (size_t j = 0; j < flavours.size(); ++j) {
                items.clear();
                for (int i = 0; i < n_tensors; ++i)
                    if (numels[i] != 0 && flavour_of[class_of[i]] == (int)j) {
                        items.push_back(tensor_item(tensors, numels, i, flavours[j].grad_f32));
                        items.back().cls = class_of[i];
                    }
                const Flavour& f = flavours[j];
                int rc = for_each_tensor_batch(items, tensors, -1, kLaunchClasses,
                                               [&](const auto& b, dim3 grid, const BatchClasses& bc) {
                    ConstsBatch cb;
                    memset(&cb, 0, sizeof(cb));
                    for (int q = 0; q < bc.n; ++q) cb.c[q] = consts[bc.of[q]];
                    if (f.arith == PS_ARITH_TORCH)
                        launch_tensors_each_arith<PS_ARITH_TORCH>(b, grid, cb, f, nt, s);
                    else
                        launch_tensors_each_arith<PS_ARITH_OPERATOR>(b, grid, cb, f, nt, s);
                }, f.grad_f32);
                if (rc) return rc;
            }
            return 0;
        }

        // ---- device-decided: the step numbers (adam_step + 1 + d), the loss scale and the operator object live on
        // the device.  The host knows how the calls relate to one another (IncrementStep, cpu_adam.h:143-162, looks
        // only at differences between consecutive calls), which leaves three kinds of operator call and one
        // torch call; the device turns each distinct one into constants.
        ClassTable<PlanClass> table_of_classes;
        const std::vector<PlanClass>& classes = table_of_classes.records;
        const std::vector<int>& class_keys = table_of_classes.arith;  // class_key(arithmetic, binary32 gradients)
        std::vector<int> class_wd;
        int prev_class = -1;  // of the previous operator call
        int last_operator = -1;
        for (int i = 0; i < n_tensors; ++i) {
            const ps_tensor_call& e = each[i];
            const int arith = arith_of(i);
            PlanClass k;
            memset(&k, 0, sizeof(k));
            k.lr = e.lr, k.beta1 = e.beta1, k.beta2 = e.beta2, k.eps = e.eps, k.wd = e.weight_decay;
            k.d = e.step;
            k.prev = -1;
            if (arith == PS_ARITH_TORCH) {
                k.mode = PLAN_TORCH;
            } else if (prev_class < 0) {
                k.mode = PLAN_FIRST;  // continues the product only if the object, as the last clean step left it, allows
            } else {
                const PlanClass& q = classes[prev_class];
                const bool same_betas = (float)q.beta1 == (float)e.beta1 && (float)q.beta2 == (float)e.beta2;
                if (same_betas && e.step == q.d + 1) {
                    k.mode = PLAN_MUL;
                    k.prev = prev_class;
                } else {
                    k.mode = PLAN_POW;
                }
            }
            if (grad_f32_of(i)) k.mode |= PLAN_GRAD_F32;
            const int c = table_of_classes.intern(k, class_key(arith, grad_f32_of(i)));
            if (c == (int)class_wd.size()) class_wd.push_back(wd_mode_of(arith, e.weight_decay, o->adamw));
            class_of[i] = c;
            if (arith != PS_ARITH_TORCH) prev_class = last_operator = c;
        }
        PlannedConsts* table = static_cast<PlannedConsts*>(d_workspace);
        const int n_classes = (int)classes.size();
        auto plan_args = [&](auto& pb, int first) {
            constexpr int N = sizeof(pb.k) / sizeof(pb.k[0]);
            memset(&pb, 0, sizeof(pb));
            PlanArgs pa;
            memset(&pa, 0, sizeof(pa));
            pa.n = std::min(N, n_classes - first);
            for (int j = 0; j < pa.n; ++j) pb.k[j] = classes[first + j];
            pa.grad_clamp = o->grad_clamp;
            pa.adamw = o->adamw ? 1 : 0;
            pa.bias_correction = bias ? 1 : 0;
            pa.first_class = first;
            pa.is_last_launch = first + N >= n_classes;
            pa.last_operator_class = last_operator;
            if (last_operator >= 0) {
                pa.last_d = classes[last_operator].d;
                pa.last_beta1 = (float)classes[last_operator].beta1;
                pa.last_beta2 = (float)classes[last_operator].beta2;
            }
            return pa;
        };
        Closing closing{};
        const Closing* closes = nullptr;
        if (whole && opens_with_plan(*whole, n_classes, class_keys, tensors, numels, n_tensors)) {
            closing = Closing{d_state, whole->scratch, whole->log, whole->log_capacity, whole->operator_calls};
            closes = &closing;
            PlanBatchOf<kOpenClasses> pb;
            const PlanArgs pa = plan_args(pb, 0);
            const ChunkList& a = whole->probed;
            ProbeList list;
            memset(&list, 0, sizeof(list));
            size_t longest = 0;
            for (int i = 0; i < a.n_chunks; ++i) {
                list.h[i] = a.chunks[i].param_fp16;
                list.n[i] = (uint32_t)a.numel_of(i);
                longest = std::max(longest, a.numel_of(i));
            }
            const dim3 grid((unsigned)((longest + kScanTile - 1) / kScanTile), (unsigned)a.n_chunks);
            with_hint(elements(a) > kScanKeepElements, [&](auto hint) {
                constexpr bool NT = decltype(hint)::value;
                hipLaunchKernelGGL((open_planned_kernel<NT>), with_first<NT>(grid), dim3(kScanBlock), kScanLdsBytes, s, list, pb, pa, d_state,
                                   whole->scratch, table, probe_keeps(a));
            });
            PS_HIP(hipGetLastError());
        } else {
            if (whole)
                if (int rc = ps_overflow_scan_chunks(whole->probed.chunks, whole->probed.n_chunks, whole->probed.chunk_numel, whole->probed.used, d_state, stream))
                    return rc;
            for (int first = 0; first < n_classes || first == 0; first += kPlanBatch) {
                PlanBatch pb;
                const PlanArgs pa = plan_args(pb, first);
                hipLaunchKernelGGL(plan_consts_kernel, dim3(1), dim3(64), 0, s, pb, pa, d_state, table);
                PS_HIP(hipGetLastError());
                if (n_classes == 0) break;
            }
        }
        // One pass of launches per (arithmetic, weight-decay form); inside it, tensors of any class.  A launch names
        // its tensors' classes in 16 bits, relative to the window of 65536 records it is handed.
        constexpr int kWindow = 1 << 16;
        std::vector<TensorItem> items;
        for (int window = 0; window < n_classes; window += kWindow) {
            for (int key : {class_key(PS_ARITH_OPERATOR, false), class_key(PS_ARITH_TORCH, false),
                            class_key(PS_ARITH_OPERATOR, true), class_key(PS_ARITH_TORCH, true)}) {
                const bool grad_f32 = key_grad_f32(key);
                for (int wd_mode : {WD_NONE, WD_L2, WD_DECOUPLED}) {
                    items.clear();
                    for (int i = 0; i < n_tensors; ++i) {
                        const int k = class_of[i];
                        if (numels[i] == 0 || k < window || k >= window + kWindow) continue;
                        if (class_keys[k] != key || class_wd[k] != wd_mode) continue;
                        items.push_back(tensor_item(tensors, numels, i, grad_f32));
                        items.back().cls = k - window;
                    }
                    if (items.empty()) continue;
                    int rc = for_each_tensor_batch(items, tensors, -1, 0,
                                                   [&](const auto& b, dim3 grid, const BatchClasses&) {
                        if (key_arith(key) == PS_ARITH_TORCH)
                            launch_tensors_planned_arith<PS_ARITH_TORCH>(b, grid, wd_mode, grad_f32, table + window, d_state, closes, nt, s);
                        else
                            launch_tensors_planned_arith<PS_ARITH_OPERATOR>(b, grid, wd_mode, grad_f32, table + window, d_state, closes, nt, s);
                        closing.st = nullptr;  // the first launch closes the step
                    }, grad_f32);
                    if (rc) return rc;
                }
            }
        }
        if (whole && !closes) return ps_scaler_update(d_state, PS_FLAG_FROM_DEVICE, whole->log, whole->log_capacity, whole->operator_calls, stream);
        return 0;
    } catch (const std::exception&) {  // nothing may throw across the boundary
        return fail(PS_ERR_BAD_ARG, "no host memory for a list of %d tensors", n_tensors);
    }
}

}  // namespace

int ps_adam_step_tensors_each(int optimizer_id, int bias_correction, const ps_chunk* tensors,
                              const size_t* numels, const ps_tensor_call* each, int n_tensors,
                              double loss_scale, ps_step_state* d_state, void* d_workspace,
                              size_t workspace_bytes, ps_stream_t stream)
{
    return step_tensors_each(optimizer_id, bias_correction, tensors, numels, each, n_tensors, loss_scale, d_state, d_workspace, workspace_bytes,
                             nullptr, stream);
}

int ps_adam_step_tensors_dynamic(int optimizer_id, int bias_correction, const ps_chunk* chunks, int n_chunks, size_t chunk_numel,
                                 const size_t* used_numel, const ps_chunk* tensors, const size_t* numels, const ps_tensor_call* each,
                                 int n_tensors, ps_step_state* d_state, ps_scale_record* d_log, int64_t log_capacity, int64_t operator_calls,
                                 void* d_workspace, size_t workspace_bytes, void* d_scratch, size_t scratch_bytes, ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (d_log != nullptr && log_capacity <= 0)
        return fail(PS_ERR_BAD_ARG, "log_capacity must be positive when d_log is given");
    if (operator_calls < 0) return fail(PS_ERR_BAD_ARG, "operator_calls = %lld is negative", (long long)operator_calls);
    if (int rc = check_scratch(d_scratch, scratch_bytes)) return rc;
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, used_numel, kScanTile, true)) return rc;
    const WholeStep whole{a, static_cast<StepScratch*>(d_scratch), d_log, log_capacity, operator_calls};
    return step_tensors_each(optimizer_id, bias_correction, tensors, numels, each, n_tensors, -1.0, d_state, d_workspace, workspace_bytes, &whole, stream);
}

int ps_tensors_at_once(const ps_chunk* chunks, int n_chunks, size_t chunk_numel, const size_t* used_numel, const ps_chunk* tensors,
                       const size_t* numels, int n_tensors)
{
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, used_numel, kScanTile, true)) return rc;
    if (int rc = check_tensor_list(tensors, numels, n_tensors)) return rc;
    try {
        return lists_open_with_plan(a, tensors, numels, n_tensors) ? 1 : 0;
    } catch (const std::exception&) {  // nothing may throw across the boundary
        return fail(PS_ERR_BAD_ARG, "no host memory for a list of %d tensors", n_tensors);
    }
}

int ps_restore_fp16_chunks(const ps_chunk* chunks, int n_chunks, size_t chunk_numel,
                           const ps_step_state* d_state, ps_stream_t stream)
{
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, nullptr, kTile)) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return for_each_batch(a, [&](const ChunkBatch& b, dim3 grid, int) {
        hipLaunchKernelGGL(restore_chunks_kernel, grid, dim3(kBlock), 0, s, b, d_state);
    });
}

int ps_cast_fp32_to_fp16(const float* d_src, uint16_t* d_dst, size_t numel, ps_stream_t stream)
{
    if (numel == 0) return 0;
    if (!d_src || !d_dst) return fail(PS_ERR_BAD_ARG, "ps_cast_fp32_to_fp16: NULL pointer");
    size_t n_tiles = (numel + kTile - 1) / kTile;
    hipLaunchKernelGGL(cast_kernel, dim3(grid_1d(n_tiles, kBlock)), dim3(kBlock), 0,
                       static_cast<hipStream_t>(stream), CastArgs{d_src, d_dst, numel, n_tiles});
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_adam_step_hybrid(int optimizer_id, size_t step, double lr, double beta1, double beta2,
                        double epsilon, double weight_decay, int bias_correction,
                        const ps_chunk* chunks, int n_chunks, const ps_chunk* host_chunks,
                        int n_host_chunks, size_t chunk_numel, const size_t* used_numel,
                        const ps_chunk* staging, int n_slots, const ps_call_pattern* calls,
                        double loss_scale, const ps_step_state* d_state, ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (n_chunks < 0) return fail(PS_ERR_BAD_ARG, "n_chunks = %d is negative", n_chunks);
    ChunkList resident, host;
    if (int rc = make_chunk_list(resident, chunks, n_chunks, chunk_numel, used_numel, kTile)) return rc;
    if (int rc = make_chunk_list(host, host_chunks, n_host_chunks, chunk_numel, used_numel ? used_numel + n_chunks : nullptr,
                                 kTile, false, "host chunk"))
        return rc;
    std::unique_ptr<bool[]> fp16_in_hbm(new (std::nothrow) bool[n_host_chunks > 0 ? n_host_chunks : 1]);
    if (!fp16_in_hbm) return fail(PS_ERR_BAD_ARG, "no host memory for a list of %d host chunks", n_host_chunks);
    if (n_host_chunks > 0) {
        if (int rc = check_slots(staging, n_slots, true, false)) return rc;
        bool any_on_host = false;
        if (int rc = fp16_payloads_in_hbm(host_chunks, n_host_chunks, fp16_in_hbm.get(), &any_on_host)) return rc;
        if (any_on_host)
            if (int rc = check_slots(staging, n_slots, true, true)) return rc;
    }
    // Resident chunks take the optimizer's arithmetic, streamed host chunks the operator's (the
    // reference updates those with the operator).  The operator object goes through the calls of
    // the pattern (over both lists), and only if the operator's arithmetic is used at all.
    const int arith = o->arith;
    Calls k;
    if (int rc = make_calls(k, calls, (int64_t)n_chunks + n_host_chunks, chunk_numel)) return rc;
    if (arith == PS_ARITH_TORCH && k.first_chunk >= 0 && k.first_chunk < n_chunks)
        return fail(PS_ERR_BAD_ARG, "calls->first_chunk = %lld names a resident chunk, which the torch arithmetic "
                    "never hands to the operator", (long long)k.first_chunk);
    StepConsts c_resident, c_host;
    const GatedArgs ga = gated_args(*o, lr, epsilon, weight_decay, bias_correction, k.n_calls);
    if (d_state == nullptr) {
        const HyperParams hp{lr, beta1, beta2, epsilon, weight_decay, loss_scale, bias_correction != 0};
        if (arith == PS_ARITH_OPERATOR || n_host_chunks > 0) c_host = operator_step_consts(*o, step, hp, k.n_calls);
        c_resident = arith == PS_ARITH_TORCH ? torch_step_consts(*o, step, hp) : c_host;
        if (!zeros_are_a_fixed_point(c_resident)) resident.used = nullptr;
        if (n_host_chunks > 0 && !zeros_are_a_fixed_point(c_host)) host.used = nullptr;
    } else {
        // Streamed chunks move only their used part over the link, so whether their padding may be left alone has
        // to be known here, from the host's numbers (the kernel's own check, on the device-resident scalars, stays
        // in force for the resident chunks): a positive eps and finite scalars, betas below one as floats.
        const bool plain = (float)epsilon > 0.0f && std::isfinite((float)lr) && std::isfinite((float)weight_decay) &&
                           std::isfinite((float)epsilon) && (float)beta1 < 1.0f && (float)beta2 < 1.0f;
        if (!plain) host.used = nullptr;
    }
    hipStream_t caller = static_cast<hipStream_t>(stream);
    bool stream_host = false;
    for (int i = 0; i < n_host_chunks; ++i) stream_host = stream_host || host.numel_of(i) > 0;
    Pipeline* p = nullptr;
    std::unique_lock<std::mutex> turn;
    bool in_place = false;
    if (stream_host) {
        if (n_host_chunks <= kMaxInPlaceChunks && in_place_pays(host, fp16_in_hbm.get(), resident))
            if (int rc = mapped_in_place(host_chunks, n_host_chunks, &in_place)) return rc;
        if (int rc = get_pipeline(&p)) return rc;
        turn = std::unique_lock<std::mutex>(p->in_use);
        // the resident chunks' kernels, queued next on the caller's stream, do NOT hold the copies back
        if (int rc = p->begin(caller)) return rc;
    }
    // (beside host chunks the link sets the pace, and 11 workgroups per CU here leave less room for theirs: 17.97 -> 18.10 ms)
    const bool nt = !stream_host && streams(resident, d_state != nullptr);
    int rc = for_each_batch(resident, [&](const ChunkBatch& b, dim3 grid, int first) {
        const FirstCall fc = k.in_batch(first, (int)grid.y);
        if (d_state == nullptr)
            launch_adam_batch(arith, b, grid, c_resident, fc, nt, caller);
        else
            launch_gated_batch(arith, b, grid, chunk_numel, ga, fc, d_state, nt, caller);
    });
    if (!stream_host) return rc;

    auto stream_chunk = [&](int k_host) -> int {
        const size_t numel = host.numel_of(k_host);
        if (numel == 0) return 0;
        const size_t b32 = numel * sizeof(float), b16 = numel * sizeof(uint16_t);
        const int s = k_host % n_slots;
        const ps_chunk& h = host_chunks[k_host];
        ps_chunk d = staging[s];
        // a fp16 payload that already lives in HBM is read and written in place: 12 instead of
        // 14 bytes per element cross the link in each direction
        const bool stage_fp16 = !fp16_in_hbm[k_host];
        if (!stage_fp16) d.param_fp16 = h.param_fp16;
        // the slot is free once its previous occupant has been written back
        if (p->slot_used[s]) PS_HIP(hipStreamWaitEvent(p->h2d, p->d2h_done[s], 0));
        if (stage_fp16)
            PS_HIP(hipMemcpyAsync(d.param_fp16, h.param_fp16, b16, hipMemcpyHostToDevice, p->h2d));
        PS_HIP(hipMemcpyAsync(d.param_fp32, h.param_fp32, b32, hipMemcpyHostToDevice, p->h2d));
        PS_HIP(hipMemcpyAsync(d.exp_avg, h.exp_avg, b32, hipMemcpyHostToDevice, p->h2d));
        PS_HIP(hipMemcpyAsync(d.exp_avg_sq, h.exp_avg_sq, b32, hipMemcpyHostToDevice, p->h2d));
        PS_HIP(hipEventRecord(p->h2d_done[s], p->h2d));

        PS_HIP(hipStreamWaitEvent(p->compute, p->h2d_done[s], 0));
        ChunkBatch b;
        memset(&b, 0, sizeof(b));
        b.c[0] = d;
        b.n[0] = numel;
        dim3 grid((unsigned)((numel + kTile - 1) / kTile), 1);
        const FirstCall fc = k.in_batch((int64_t)n_chunks + k_host, 1);
        if (d_state == nullptr)
            launch_adam_batch(PS_ARITH_OPERATOR, b, grid, c_host, fc, false, p->compute);
        else  // the staged copy ends at `numel`: nothing behind it for the kernel to decide about
            launch_gated_batch(PS_ARITH_OPERATOR, b, grid, numel, ga, fc, d_state, false, p->compute);
        PS_HIP(hipGetLastError());
        PS_HIP(hipEventRecord(p->compute_done[s], p->compute));

        PS_HIP(hipStreamWaitEvent(p->d2h, p->compute_done[s], 0));
        // (on a device-skipped step fp32 param / m / v come back unchanged; copying them anyway
        // keeps the host free of any knowledge of the flag)
        if (stage_fp16)
            PS_HIP(hipMemcpyAsync(h.param_fp16, d.param_fp16, b16, hipMemcpyDeviceToHost, p->d2h));
        PS_HIP(hipMemcpyAsync(h.param_fp32, d.param_fp32, b32, hipMemcpyDeviceToHost, p->d2h));
        PS_HIP(hipMemcpyAsync(h.exp_avg, d.exp_avg, b32, hipMemcpyDeviceToHost, p->d2h));
        PS_HIP(hipMemcpyAsync(h.exp_avg_sq, d.exp_avg_sq, b32, hipMemcpyDeviceToHost, p->d2h));
        PS_HIP(hipEventRecord(p->d2h_done[s], p->d2h));
        p->slot_used[s] = true;
        return 0;
    };
    if (in_place) {
        if (rc == 0)
            rc = for_each_batch(host, [&](const ChunkBatch& b, dim3 grid, int first) {
                const FirstCall fc = k.in_batch((int64_t)n_chunks + first, (int)grid.y);
                if (d_state == nullptr)
                    launch_adam_batch(PS_ARITH_OPERATOR, b, grid, c_host, fc, false, p->compute);
                else  // chunk_numel 0: as on a staged copy, what lies behind the used part is not looked at
                    launch_gated_batch(PS_ARITH_OPERATOR, b, grid, 0, ga, fc, d_state, false, p->compute);
            });
    } else {
        for (int i = 0; i < n_host_chunks && rc == 0; ++i) rc = stream_chunk(i);
    }
    // later work on the caller's stream sees every chunk written back (also if queuing stopped half way, or never
    // started because a resident launch failed: the side streams already wait on the caller, the caller must wait
    // on them)
    const int joined = p->join(caller);
    return rc ? rc : joined;
}

int ps_overflow_scan_host_chunks(const ps_chunk* host_chunks, int n_chunks, size_t chunk_numel,
                                 const size_t* used_numel, const ps_chunk* staging, int n_slots,
                                 ps_step_state* d_state, ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    ChunkList a;
    if (int rc = make_chunk_list(a, host_chunks, n_chunks, chunk_numel, used_numel, kScanTile, true, "host chunk")) return rc;
    if (n_chunks == 0 || chunk_numel == 0) return 0;
    std::unique_ptr<bool[]> fp16_in_hbm(new (std::nothrow) bool[n_chunks]);
    if (!fp16_in_hbm) return fail(PS_ERR_BAD_ARG, "no host memory for a list of %d host chunks", n_chunks);
    bool any_on_host = false;
    if (int rc = fp16_payloads_in_hbm(host_chunks, n_chunks, fp16_in_hbm.get(), &any_on_host)) return rc;
    hipStream_t caller = static_cast<hipStream_t>(stream);
    auto tiles_of = [&](int k) { return (a.numel_of(k) + kScanTile - 1) / kScanTile; };
    // fp16 payloads that live in HBM are probed in place on the caller's stream
    for (int k = 0; k < n_chunks; ++k) {
        if (!fp16_in_hbm[k] || a.numel_of(k) == 0) continue;
        hipLaunchKernelGGL(scan_f16_kernel, dim3(grid_1d(tiles_of(k), kScanBlock)), dim3(kScanBlock), kScanLdsBytes, caller,
                           host_chunks[k].param_fp16, a.numel_of(k), tiles_of(k), d_state);
        PS_HIP(hipGetLastError());
    }
    any_on_host = false;
    for (int k = 0; k < n_chunks; ++k) any_on_host = any_on_host || (!fp16_in_hbm[k] && a.numel_of(k) > 0);
    if (!any_on_host) return 0;
    if (int rc = check_slots(staging, n_slots, false, true)) return rc;
    Pipeline* p = nullptr;
    if (int rc = get_pipeline(&p)) return rc;
    std::lock_guard<std::mutex> turn(p->in_use);
    if (int rc = p->begin(caller)) return rc;
    int streamed = 0;
    auto stream_chunk = [&](int k) -> int {
        const int s = streamed++ % n_slots;
        if (p->slot_used[s]) PS_HIP(hipStreamWaitEvent(p->h2d, p->compute_done[s], 0));
        PS_HIP(hipMemcpyAsync(staging[s].param_fp16, host_chunks[k].param_fp16, a.numel_of(k) * sizeof(uint16_t),
                              hipMemcpyHostToDevice, p->h2d));
        PS_HIP(hipEventRecord(p->h2d_done[s], p->h2d));
        PS_HIP(hipStreamWaitEvent(p->compute, p->h2d_done[s], 0));
        hipLaunchKernelGGL(scan_f16_kernel, dim3(grid_1d(tiles_of(k), kScanBlock)), dim3(kScanBlock), kScanLdsBytes, p->compute,
                           staging[s].param_fp16, a.numel_of(k), tiles_of(k), d_state);
        PS_HIP(hipGetLastError());
        PS_HIP(hipEventRecord(p->compute_done[s], p->compute));
        p->slot_used[s] = true;
        return 0;
    };
    int rc = 0;
    for (int k = 0; k < n_chunks && rc == 0; ++k)
        if (!fp16_in_hbm[k] && a.numel_of(k) > 0) rc = stream_chunk(k);
    const int joined = p->join(caller);
    return rc ? rc : joined;
}

int ps_state_init(ps_step_state* d_state, double init_scale, int init_is_int, double scale_factor,
                  int factor_is_int, int64_t scale_window, double min_scale, int min_is_int,
                  int delayed_shift, int consecutive_hysteresis, double beta1, double beta2,
                  ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (scale_window <= 0)
        return fail(PS_ERR_BAD_ARG, "scale_window = %lld must be positive", (long long)scale_window);
    ps_step_state s;
    memset(&s, 0, sizeof(s));
    s.cur_scale = init_scale;
    s.scale_is_int = init_is_int != 0;
    s.scale_factor = scale_factor;
    s.factor_is_int = factor_is_int != 0;
    s.min_scale = min_scale;
    s.min_is_int = min_is_int != 0;
    s.cur_iter = 0;
    s.last_overflow_iter = -1;
    s.scale_window = scale_window;
    s.delayed_shift = delayed_shift;
    s.cur_hysteresis = delayed_shift;
    s.consecutive_hysteresis = consecutive_hysteresis != 0;
    s.beta1 = (float)beta1;
    s.beta2 = (float)beta2;
    // Adam_Optimizer starts with beta^t = 1 and step 0; the first update multiplies once.
    s.operator_step = 0;
    s.operator_beta1 = s.beta1;
    s.operator_beta2 = s.beta2;
    s.beta1_t_cur = 1.0f;
    s.beta2_t_cur = 1.0f;
    s.beta1_t_next = 1.0f * s.beta1;
    s.beta2_t_next = 1.0f * s.beta2;
    // a second call of step 1 finds _step + 1 = 2 != 1 and evaluates pow(beta, 1)
    s.beta1_t_rest = (float)std::pow((double)s.beta1, 1.0);
    s.beta2_t_rest = (float)std::pow((double)s.beta2, 1.0);
    s.beta1_f64 = beta1;
    s.beta2_f64 = beta2;
    s.bias_correction1_next = 1.0 - std::pow(beta1, 1.0);
    s.bias_correction2_next = 1.0 - std::pow(beta2, 1.0);
    hipLaunchKernelGGL(state_init_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                       d_state, s);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_state_seed_step(ps_step_state* d_state, int64_t adam_step, double beta1, double beta2,
                       int fresh_operator, ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (adam_step < 0) return fail(PS_ERR_BAD_ARG, "adam_step is negative");
    SeedArgs a;
    a.adam_step = adam_step;
    a.beta1 = (float)beta1;
    a.beta2 = (float)beta2;
    // what a call for step adam_step + 1 gets when it cannot continue a running product; whether the
    // first call of that step can is decided on the device, where the operator object's state lives
    a.b1t_rest = (float)std::pow((double)a.beta1, (double)(adam_step + 1));
    a.b2t_rest = (float)std::pow((double)a.beta2, (double)(adam_step + 1));
    a.fresh_operator = fresh_operator != 0;
    a.beta1_f64 = beta1;
    a.beta2_f64 = beta2;
    a.bc1_next = 1.0 - std::pow(beta1, (double)(adam_step + 1));
    a.bc2_next = 1.0 - std::pow(beta2, (double)(adam_step + 1));
    hipLaunchKernelGGL(state_seed_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                       d_state, a);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_state_set_scaler(ps_step_state* d_state, double cur_scale, int scale_is_int,
                        int64_t cur_iter, int64_t last_overflow_iter, int cur_hysteresis,
                        ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    hipLaunchKernelGGL(state_set_scaler_kernel, dim3(1), dim3(64), 0,
                       static_cast<hipStream_t>(stream), d_state, cur_scale, scale_is_int, cur_iter,
                       last_overflow_iter, cur_hysteresis);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_overflow_scan(const uint16_t* d_grads_fp16, size_t numel, ps_step_state* d_state,
                     ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (numel == 0) return 0;
    if (!d_grads_fp16) return fail(PS_ERR_BAD_ARG, "d_grads_fp16 is NULL");
    size_t n_tiles = (numel + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(scan_f16_kernel, dim3(grid_1d(n_tiles, kScanBlock)), dim3(kScanBlock), kScanLdsBytes,
                       static_cast<hipStream_t>(stream), d_grads_fp16, numel, n_tiles, d_state);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_overflow_scan_f32(const float* d_grads_fp32, size_t numel, ps_step_state* d_state,
                         ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (numel == 0) return 0;
    if (!d_grads_fp32) return fail(PS_ERR_BAD_ARG, "d_grads_fp32 is NULL");
    size_t n_tiles = (numel + kScanTileF32 - 1) / kScanTileF32;
    hipLaunchKernelGGL(scan_f32_kernel, dim3(grid_1d(n_tiles, kScanBlock)), dim3(kScanBlock), kScanLdsBytes,
                       static_cast<hipStream_t>(stream), d_grads_fp32, numel, n_tiles, d_state);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_overflow_scan_chunks(const ps_chunk* chunks, int n_chunks, size_t chunk_numel,
                            const size_t* used_numel, ps_step_state* d_state, ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, used_numel, kScanTile, true)) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool nt = elements(a) > kScanKeepElements;
    EvenList e;
    if (even_list(a, kMaxEvenElementsGated, &e, true)) {
        with_hint(nt, [&](auto hint) {
            hipLaunchKernelGGL((scan_even_chunks_kernel<decltype(hint)::value>), even_grid(e, kScanTile), dim3(kScanBlock), kScanLdsBytes, s,
                               e.first.param_fp16, e.stride, e.numel, e.last, e.short_by, d_state, probe_keeps(a));
        });
        PS_HIP(hipGetLastError());
        return 0;
    }
    return for_each_batch(a, [&](const ChunkBatch& b, dim3 grid, int first) {
        with_hint(nt, [&](auto hint) {
            hipLaunchKernelGGL((scan_chunks_kernel<decltype(hint)::value>), grid, dim3(kScanBlock), kScanLdsBytes, s, b, d_state,
                               first ? 0 : probe_keeps(a));
        });
    });
}

int ps_overflow_scan_chunks_noalloc(const ps_chunk* chunks, int n_chunks, size_t chunk_numel,
                                    uint32_t* d_flag, ps_stream_t stream)
{
    if (!d_flag) return fail(PS_ERR_BAD_ARG, "d_flag is NULL");
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, nullptr, kPartialTile)) return rc;
    const size_t tiles_per_chunk = (chunk_numel + kPartialTile - 1) / kPartialTile;
    if (n_chunks == 0 || tiles_per_chunk == 0) return 0;
    // one scratch word per workgroup of the first kernel
    const size_t max_chunks = kScratchWords / tiles_per_chunk;  // 0 when one chunk alone is too long
    if ((size_t)n_chunks > max_chunks)
        return fail(PS_ERR_BAD_ARG,
                    "%d chunks of %zu elements need %zu scratch words; this entry point holds %zu (at most %zu "
                    "elements per call): split the list or use ps_overflow_scan_chunks",
                    n_chunks, chunk_numel, (size_t)n_chunks * tiles_per_chunk, kScratchWords,
                    kScratchWords * (size_t)kPartialTile);
    uint32_t* scratch = nullptr;
    if (int rc = scratch_address(&scratch)) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    int rc = for_each_batch(a, [&](const ChunkBatch& b, dim3 grid, int first) {
        hipLaunchKernelGGL(scan_chunks_partial_kernel, grid, dim3(kPartialBlock), kScanLdsBytes, s, b,
                           scratch + (size_t)first * tiles_per_chunk);
    });
    if (rc) return rc;
    // a workgroup per 8192 words (a single one took 33 us over the 196,608 words of 24 x 64 Mi elements)
    const size_t n_words = (size_t)n_chunks * tiles_per_chunk;
    const unsigned reducers = (unsigned)std::min<size_t>((n_words + 8191) / 8192, 128);
    hipLaunchKernelGGL(scan_reduce_kernel, dim3(reducers), dim3(kReduceBlock), 0, s, scratch, n_words, d_flag);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_grads_to_chunks(const ps_grad_copy* copies, int n_copies, ps_step_state* d_state, ps_stream_t stream)
{
    if (n_copies < 0) return fail(PS_ERR_BAD_ARG, "n_copies = %d is negative", n_copies);
    if (n_copies > 0 && !copies) return fail(PS_ERR_BAD_ARG, "copies is NULL");
    for (int i = 0; i < n_copies; ++i) {
        if (copies[i].numel > 0 && (!copies[i].d_grad || !copies[i].d_slot_fp16))
            return fail(PS_ERR_BAD_ARG, "copy %d has a NULL address", i);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    int next = 0;
    size_t done = 0;  // elements of copies[next] that earlier launches have taken
    while (next < n_copies) {
        GradBatch b;
        memset(&b, 0, sizeof(b));
        memset(b.first_block, 0xFF, sizeof(b.first_block));
        size_t blocks = 0;
        int in_batch = 0;
        while (next < n_copies && in_batch < kGradBatch && blocks < kMaxCopyBlocks) {
            const ps_grad_copy& c = copies[next];
            // what is left of a gradient if that fits into the launch grid, else whole spans, and the rest in the next launch
            const size_t left = c.numel - done, room = (kMaxCopyBlocks - blocks) * kCopySpan;
            const size_t numel = std::min(left, room);
            if (numel > 0) {
                b.src[in_batch] = static_cast<const char*>(c.d_grad) + done * (c.grad_is_half ? 2 : 4);
                b.dst[in_batch] = c.d_slot_fp16 + done;
                b.numel_half[in_batch] = 2 * (uint64_t)numel + (c.grad_is_half ? 1 : 0);
                b.first_block[in_batch] = (uint32_t)blocks;
                blocks += (numel + kCopySpan - 1) / kCopySpan;
                in_batch += 1;
            }
            done += numel;
            if (done == c.numel) next += 1, done = 0;
        }
        if (in_batch == 0) continue;
        const dim3 grid((unsigned)blocks), block(kCopyBlock);
        if (in_batch == 1)
            hipLaunchKernelGGL(grad_to_chunk_kernel, grid, block, 0, s, GradCopy{b.src[0], b.dst[0], b.numel_half[0], d_state});
        else
            hipLaunchKernelGGL(grads_to_chunks_kernel, grid, block, 0, s, b, d_state);
        PS_HIP(hipGetLastError());
    }
    return 0;
}

int ps_grad_to_chunk(const void* d_grad, int grad_is_half, uint16_t* d_slot_fp16, size_t numel,
                     ps_step_state* d_state, ps_stream_t stream)
{
    if (numel == 0) return 0;
    if (!d_grad || !d_slot_fp16) return fail(PS_ERR_BAD_ARG, "ps_grad_to_chunk: NULL pointer");
    const ps_grad_copy c{d_grad, d_slot_fp16, numel, grad_is_half != 0};
    return ps_grads_to_chunks(&c, 1, d_state, stream);
}

int ps_scaler_update(ps_step_state* d_state, int flag_mode, ps_scale_record* d_log,
                     int64_t log_capacity, int64_t operator_calls, ps_stream_t stream)
{
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (flag_mode < 0 || flag_mode > 2) return fail(PS_ERR_BAD_ARG, "flag_mode = %d", flag_mode);
    if (d_log != nullptr && log_capacity <= 0)
        return fail(PS_ERR_BAD_ARG, "log_capacity must be positive when d_log is given");
    if (operator_calls < 0) return fail(PS_ERR_BAD_ARG, "operator_calls = %lld is negative", (long long)operator_calls);
    hipLaunchKernelGGL(scaler_update_kernel, dim3(1), dim3(64), 0,
                       static_cast<hipStream_t>(stream), d_state, flag_mode, d_log, log_capacity,
                       operator_calls);
    PS_HIP(hipGetLastError());
    return 0;
}

int ps_adam_step_chunks_dynamic_scratch(int optimizer_id, double lr, double epsilon, double weight_decay, int bias_correction,
                                        const ps_chunk* chunks, int n_chunks, size_t chunk_numel, const size_t* used_numel,
                                        const ps_call_pattern* calls, int probe, ps_step_state* d_state, ps_scale_record* d_log,
                                        int64_t log_capacity, int64_t operator_calls, void* d_scratch, size_t scratch_bytes,
                                        ps_stream_t stream)
{
    auto o = find_opt(optimizer_id);
    if (!o) return fail(PS_ERR_UNKNOWN_ID, "optimizer id %d was never created", optimizer_id);
    if (!d_state) return fail(PS_ERR_BAD_ARG, "d_state is NULL");
    if (d_log != nullptr && log_capacity <= 0)
        return fail(PS_ERR_BAD_ARG, "log_capacity must be positive when d_log is given");
    if (operator_calls < 0) return fail(PS_ERR_BAD_ARG, "operator_calls = %lld is negative", (long long)operator_calls);
    if (int rc = check_scratch(d_scratch, scratch_bytes)) return rc;
    ChunkList a;
    if (int rc = make_chunk_list(a, chunks, n_chunks, chunk_numel, used_numel, kTile)) return rc;
    Calls k;
    if (int rc = make_calls(k, calls, n_chunks, chunk_numel)) return rc;
    StepScratch* const scratch = static_cast<StepScratch*>(d_scratch);
    size_t longest = 0;
    for (int i = 0; i < n_chunks; ++i) longest = std::max(longest, a.numel_of(i));
    const size_t tiles = (longest + kTile - 1) / kTile;
    if (n_chunks <= kBatch && tiles > 0 && tiles <= (scratch ? kSmallTiles : kSmallTilesAlone) / n_chunks) {
        const GatedArgs ga = gated_args(*o, lr, epsilon, weight_decay, bias_correction, k.n_calls);
        const uint32_t scans = (uint32_t)((longest + kSmallScan - 1) / kSmallScan);
        auto reciprocal = [](size_t n) { return (uint32_t)((((uint64_t)1 << 32) + n - 1) / n); };
        const SmallStep step{(uint32_t)tiles, (uint32_t)(tiles * n_chunks), reciprocal(tiles), scans, probe ? scans * n_chunks : 0, reciprocal(scans),
                             chunk_numel, d_log, log_capacity, operator_calls};
        const int arith = o->arith;
        hipStream_t s = static_cast<hipStream_t>(stream);
        EvenList e;
        if (even_list(a, kMaxEvenElementsGated, &e)) {
            launch_small_step(arith, e, step, ga, k.in_batch(0, n_chunks), d_state, scratch, s);
            PS_HIP(hipGetLastError());
            return 0;
        }
        return for_each_batch(a, [&](const ChunkBatch& b, dim3, int) {
            launch_small_step(arith, b, step, ga, k.in_batch(0, n_chunks), d_state, scratch, s);
        });
    }
    // Two launches: lists of evenly spaced chunks, and other lists below the line from which they stream past the caches.  (Beyond it the update's
    // waves with descriptors, which read the copy behind them, lose what the third launch costs: 8 x 64 Mi elements in three / two
    // 2423 / 2431 us, a skipped step 614 / 623.)
    EvenList e;
    const bool even = even_list(a, kMaxEvenElementsGated, &e);
    if (probe && scratch && tiles > 0 && tiles <= kMaxGridX - kInFront<true> && (even || (n_chunks <= kBatch && elements(a) < kStreamElementsGated))) {
        const GatedArgs ga = gated_args(*o, lr, epsilon, weight_decay, bias_correction, k.n_calls);
        const Closing cl{d_state, scratch, d_log, log_capacity, operator_calls};
        hipStream_t s = static_cast<hipStream_t>(stream);
        const bool torch = o->arith == PS_ARITH_TORCH;
        const FirstCall fc = torch ? kNoFirstCall : k.in_batch(0, n_chunks);
        if (even) {
            const bool nt = streams(a, true);
            with_hint(elements(a) > kScanKeepElements, [&](auto hint) {
                hipLaunchKernelGGL((open_even_chunks_kernel<decltype(hint)::value>), with_first<decltype(hint)::value>(even_grid(e, kScanTile)), dim3(kScanBlock), kScanLdsBytes, s,
                                   e.first.param_fp16, e.stride, e.numel, e.last, e.short_by, d_state, scratch, probe_keeps(a));
            });
            PS_HIP(hipGetLastError());
            if (torch)
                launch_even_closing<PS_ARITH_TORCH>(e, chunk_numel, ga, fc, cl, nt, s);
            else
                launch_even_closing<PS_ARITH_OPERATOR>(e, chunk_numel, ga, fc, cl, nt, s);
            PS_HIP(hipGetLastError());
            return 0;
        }
        ChunkList probed = a;
        probed.tile = kScanTile;
        if (int rc = for_each_batch(probed, [&](const ChunkBatch& b, dim3 grid, int) {
                hipLaunchKernelGGL(open_chunks_kernel, with_first<false>(grid), dim3(kScanBlock), kScanLdsBytes, s, b, d_state, scratch);
            }))
            return rc;
        return for_each_batch(a, [&](const ChunkBatch& b, dim3 grid, int) {
            if (torch)
                launch_closing_batch<PS_ARITH_TORCH>(b, grid, chunk_numel, ga, fc, cl, s);
            else
                launch_closing_batch<PS_ARITH_OPERATOR>(b, grid, chunk_numel, ga, fc, cl, s);
        });
    }
    if (probe)
        if (int rc = ps_overflow_scan_chunks(chunks, n_chunks, chunk_numel, used_numel, d_state, stream)) return rc;
    if (int rc = ps_adam_step_chunks_gated(optimizer_id, lr, epsilon, weight_decay, bias_correction, chunks, n_chunks,
                                           chunk_numel, used_numel, calls, d_state, stream))
        return rc;
    return ps_scaler_update(d_state, PS_FLAG_FROM_DEVICE, d_log, log_capacity, operator_calls, stream);
}

int ps_adam_step_chunks_dynamic(int optimizer_id, double lr, double epsilon, double weight_decay, int bias_correction,
                                const ps_chunk* chunks, int n_chunks, size_t chunk_numel, const size_t* used_numel,
                                const ps_call_pattern* calls, int probe, ps_step_state* d_state, ps_scale_record* d_log,
                                int64_t log_capacity, int64_t operator_calls, ps_stream_t stream)
{
    return ps_adam_step_chunks_dynamic_scratch(optimizer_id, lr, epsilon, weight_decay, bias_correction, chunks, n_chunks, chunk_numel, used_numel,
                                               calls, probe, d_state, d_log, log_capacity, operator_calls, nullptr, 0, stream);
}

int ps_state_read(const ps_step_state* d_state, ps_step_state* host_out, ps_stream_t stream)
{
    if (!d_state || !host_out) return fail(PS_ERR_BAD_ARG, "ps_state_read: NULL pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    PS_HIP(hipMemcpyAsync(host_out, d_state, sizeof(ps_step_state), hipMemcpyDeviceToHost, s));
    PS_HIP(hipStreamSynchronize(s));
    return 0;
}

}  // extern "C"
