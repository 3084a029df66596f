// The kernels: fused chunk-list step (host-decided and device-gated), restore / cast, flat-tensor operator, inf/nan probe, gradient-to-chunk copy, step-state maintenance.
#ifndef PS_KERNELS_H
#define PS_KERNELS_H

#include "ps_tile.h"

namespace {

// ------------------------------------------------------- chunk-list kernels
//
// Grid: x = tile inside a chunk, y = chunk inside the batch.  Up to kBatch
// descriptors are passed BY VALUE in the kernel-argument segment.

constexpr int kBatch = 64;
struct ChunkBatch {
    ps_chunk c[kBatch];
    size_t n[kBatch];  // elements of each chunk the launch covers: the chunk's length, or less when only zeros follow
};
static_assert(sizeof(ps_chunk) == 32 && sizeof(ps_step_state) == 256 && sizeof(ps_scale_record) == 16 &&
                  sizeof(ps_call_pattern) == 32 && sizeof(ps_tensor_call) == 56,
              "layout of the boundary structs");

// What a workgroup needs before its first data load, fetched from the kernel arguments in one go.  Left to itself the
// compiler loads the length, tests it, loads the call span, tests it, and only then loads the addresses: three waits
// for scalar memory in a row in front of every tile's data loads.  The empty asm asks for all of them at once; the
// device-decided kernel had five such rounds and has three (arguments, step state, constants).  What that is worth is about
// what one run and the next differ by: both forms alternated on one box, 7207 and 7187 us for 24 x 64 Mi elements, 308 and
// 305 us for one chunk, 2602 and 2595 us for a clean device-decided step over eight, probe included; the same step on other
// boxes takes 7.10 to 7.35 ms.
struct TileSource {
    float *p32, *m32, *v32;
    uint16_t* h16;
    size_t numel;
};
__device__ __forceinline__ TileSource tile_source(const ps_chunk& c, uint64_t numel)
{
    TileSource t{c.param_fp32, c.exp_avg, c.exp_avg_sq, c.param_fp16, (size_t)numel};
    asm volatile("" : "+s"(t.p32), "+s"(t.m32), "+s"(t.v32), "+s"(t.h16), "+s"(t.numel));
    return t;
}
__device__ __forceinline__ ps_chunk as_chunk(const TileSource& t) { return ps_chunk{t.p32, t.m32, t.v32, t.h16}; }
__device__ __forceinline__ bool aligned16(const TileSource& t) { return aligned16(t.p32, t.m32, t.v32, t.h16); }
// a tile number below this one is a whole tile (lengths are below 2^34 elements: see kMaxGridX)
__device__ __forceinline__ uint32_t whole_tiles(size_t numel) { return (uint32_t)(numel / kTile); }

// The span of the step's first operator call, as seen from this workgroup's tile: wholly inside it, or cut by one of
// its ends.
struct CallSpan {
    bool here, inside, cut;
};
__device__ __forceinline__ CallSpan call_span(const FirstCall& fc, uint32_t tile)
{
    CallSpan s;
    s.here = fc.chunk == (int)blockIdx.y;
    s.inside = s.here && tile >= fc.in_lo && tile < fc.in_hi;
    s.cut = s.here && !s.inside && tile >= fc.lo_tile && tile < fc.hi_tile;
    return s;
}

// Host-decided step: all scalars arrive as kernel arguments and the
// arithmetic variant is a compile-time property of the kernel.
template <int ARITH, int WD, int UNS, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_chunks_kernel(ChunkBatch b, StepConsts c, FirstCall fc)
{
    // b.n: the host has already decided whether the zeros behind a chunk's last tensor may be left alone
    const TileSource t = tile_source(b.c[blockIdx.y], b.n[blockIdx.y]);
    const CallSpan s = call_span(fc, blockIdx.x);
    const size_t base = (size_t)blockIdx.x * kTile;
    if (blockIdx.x < whole_tiles(t.numel) && !s.cut && aligned16(t)) {
        LaneTile r;
        tile_load<false, NT>(r, t.p32, t.m32, t.v32, t.h16, base);
        tile_finish<ARITH, WD, UNS, false, NT>(c, s.inside ? c.first_step_size : c.step_size, s.inside ? c.first_bc2inv : c.bc2inv, r,
                                               t.p32, t.m32, t.v32, t.h16, base);
        return;
    }
    if (base >= t.numel) return;  // the grid is as wide as the longest chunk of the batch
    adam_tile<ARITH, WD, UNS>(c, as_chunk(t), base, t.numel, s.here ? fc.lo : 0, s.here ? fc.hi : 0);
}

// Chunks that follow one another at one distance in all four lists, all of one length but perhaps the last: what
// PatrickStarClient allocates.  Addresses, distance and lengths are 12 words (with the step state's address 14), which are
// preloaded into scalar registers, so a wave asks for its data, or for the step state, before it has waited for anything.
//
// Device time, descriptors / preloaded, host-decided: 128 K elements 2.60 / 2.36 us, 1 Mi 7.98 / 7.64, 4 Mi 23.3 / 22.7, 16 Mi
// 77.4 / 77.2; device-decided, with the probe and the scale update: 128 K 9.27 / 8.65, 1 Mi 15.4 / 13.8, 4 Mi 31.4 / 29.3, 16 Mi
// 89.6 / 87.4; 64 Mi, with the hint, 306.8 / 305.5; the probe alone 2.19 / 1.87 at 1 Mi, 6.24 / 5.85 at 16 Mi.
struct EvenChunk {
    float *p32, *m32, *v32;
    uint16_t* h16;
    size_t numel;
};
__device__ __forceinline__ EvenChunk even_chunk(float* p32, float* m32, float* v32, uint16_t* h16, uint32_t stride, uint32_t numel, uint32_t last, uint32_t short_by)
{
    const size_t at = (size_t)stride * blockIdx.y;
    return EvenChunk{p32 + at, m32 + at, v32 + at, h16 + at, (size_t)(numel - (blockIdx.y == last ? short_by : 0u))};
}

template <int ARITH, int WD, int UNS, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_even_chunks_kernel(float* p32, float* m32, float* v32, uint16_t* h16, uint32_t stride, uint32_t numel, uint32_t last,
                            uint32_t short_by, StepConsts c, FirstCall fc)
{
    const EvenChunk t = even_chunk(p32, m32, v32, h16, stride, numel, last, short_by);
    const size_t base = (size_t)blockIdx.x * kTile;
    if (blockIdx.x < whole_tiles(t.numel)) {
        LaneTile r;
        tile_load<false, NT>(r, t.p32, t.m32, t.v32, t.h16, base);
        __builtin_amdgcn_sched_barrier(0);  // the loads in front of the wait for the arguments behind the preloaded ones
        const CallSpan s = call_span(fc, blockIdx.x);
        if (!s.cut) {
            tile_finish<ARITH, WD, UNS, false, NT>(c, s.inside ? c.first_step_size : c.step_size, s.inside ? c.first_bc2inv : c.bc2inv, r, t.p32,
                                        t.m32, t.v32, t.h16, base);
            return;
        }
    }
    if (base >= t.numel) return;
    const bool here = fc.chunk == (int)blockIdx.y;
    adam_tile_scalar<ARITH, WD, UNS>(c, t.p32, t.m32, t.v32, t.h16, base, base + kTile < t.numel ? base + kTile : t.numel,
                                     here ? fc.lo : 0, here ? fc.hi : 0);
}

struct GatedArgs {
    double lr, eps, wd;  // the Python numbers; the operator's arithmetic narrows them to float
    double grad_clamp;
    int64_t n_calls;  // operator calls the reference makes in this step (its tensors); <= 1: the list is one call
    int adamw;
    int bias_correction;
};

// Device-decided step: overflow flag, loss scale and beta^t come from the
// device-resident state; a flagged step restores fp16 from fp32 instead.
// The weight-decay form is known to the host; the unscale form depends on
// the device-resident scale and is a uniform branch around the arithmetic.
// Step constants of a device-decided step, formed by every wave from the device-resident state.
// `with_first_call`: this workgroup's chunk (tensor) holds elements of the step's first operator call; every
// other workgroup is spared the second pair of bias scalars (a divide and a square root per wave).
// What a device-decided step reads from the device-resident state, fetched in one go (a handful of wide scalar
// loads issued together) instead of field by field as the arithmetic gets to them.
struct StateView {
    double cur_scale, beta1_f64, beta2_f64, bc1_next, bc2_next;
    float beta1, beta2, b1t_next, b2t_next, b1t_rest, b2t_rest;
    uint32_t overflow;
};
__device__ __forceinline__ StateView view_state(const ps_step_state* __restrict__ st)
{
    StateView s;
    s.overflow = st->overflow;
    s.cur_scale = st->cur_scale;
    s.beta1 = st->beta1;
    s.beta2 = st->beta2;
    s.b1t_next = st->beta1_t_next;
    s.b2t_next = st->beta2_t_next;
    s.b1t_rest = st->beta1_t_rest;
    s.b2t_rest = st->beta2_t_rest;
    s.beta1_f64 = st->beta1_f64;
    s.beta2_f64 = st->beta2_f64;
    s.bc1_next = st->bias_correction1_next;
    s.bc2_next = st->bias_correction2_next;
    return s;
}

template <int ARITH>
__device__ __forceinline__ StepConsts gated_consts(const GatedArgs& ga, const StateView& st, bool with_first_call)
{
    StepConsts c;
    const float clip = clamp_bound(ga.grad_clamp, st.cur_scale);
    if (ARITH == PS_ARITH_OPERATOR) {
        // The operator takes its scalars and loss_scale as C floats: the Python numbers narrow (RNE).
        // one operator call in the step: everything is that (first) call
        const bool one_call = ga.n_calls <= 1;
        const float b1t = one_call ? st.b1t_next : st.b1t_rest;
        const float b2t = one_call ? st.b2t_next : st.b2t_rest;
        finish_consts(c, (float)ga.lr, st.beta1, st.beta2, (float)ga.eps, (float)ga.wd, ga.adamw != 0, b1t, b2t,
                      ga.bias_correction != 0, (float)st.cur_scale, clip);
        if (with_first_call && !one_call)
            bias_scalars((float)ga.lr, st.b1t_next, st.b2t_next, ga.bias_correction != 0, &c.first_step_size,
                         &c.first_bc2inv);
    } else {
        const bool bc = ga.bias_correction != 0;
        torch_consts(c, ga.lr, st.beta1_f64, st.beta2_f64, ga.eps, ga.wd, ga.adamw != 0, bc ? st.bc1_next : 1.0,
                     bc ? st.bc2_next : 1.0, st.cur_scale, clip);
    }
    return c;
}

// Zeros in all four lists stay zeros under these constants (so the padding behind a chunk's last tensor need not
// be touched): the denominator sqrt(0) * bc2inv + eps is a positive number and nothing multiplies a zero by an
// infinity or a NaN.  With eps == 0 the reference's arithmetic writes 0 / 0 into the padding; then it is computed.
__host__ __device__ inline bool zeros_are_a_fixed_point(const StepConsts& c)
{
    const float s = c.step_size + c.first_step_size + c.bc2inv + c.first_bc2inv + c.wd_term + c.scale + c.beta1 +
                    c.beta2 + c.b1m + c.b2m + c.eps;
    return c.eps > 0.0f && (s - s) == 0.0f;  // every term finite (no NaN, and no infinities: inf - inf is NaN)
}

// One tile of a device-decided step, over a list with descriptors.
template <int ARITH, int WD, bool NT>
__device__ __forceinline__ void gated_tile(const TileSource& t, uint32_t tile, const CallSpan& s, size_t chunk_numel, const GatedArgs& ga,
                                           const FirstCall& fc, const StateView& sv)
{
    const size_t base = (size_t)tile * kTile;
    if (__builtin_expect(sv.overflow, 0)) {
        if (restore_leader(tile)) restore_tiles<NT>(t.p32, t.h16, base, t.numel);  // RNE(0) = 0 is already there
        return;
    }
    if (tile < whole_tiles(t.numel) && !s.cut && aligned16(t)) {
        LaneTile r;
        tile_load<false, NT>(r, t.p32, t.m32, t.v32, t.h16, base);
        const StepConsts c = gated_consts<ARITH>(ga, sv, s.here);
        tile_finish<ARITH, WD, UNSCALE_RUNTIME, false, NT>(c, s.inside ? c.first_step_size : c.step_size, s.inside ? c.first_bc2inv : c.bc2inv, r,
                                                t.p32, t.m32, t.v32, t.h16, base);
        return;
    }
    size_t numel = t.numel;  // what lies behind it is zeros in all four lists
    if (base + kTile > numel && numel < chunk_numel) {
        // a tile that reaches into the padding: leave the zeros alone only if they are a fixed point of this step
        if (!zeros_are_a_fixed_point(gated_consts<ARITH>(ga, sv, s.here))) numel = chunk_numel;
    }
    if (base >= numel) return;
    adam_tile_late_consts<ARITH, WD, UNSCALE_RUNTIME>([&]() { return gated_consts<ARITH>(ga, sv, s.here); }, as_chunk(t), base,
                                                      numel, s.here ? fc.lo : 0, s.here ? fc.hi : 0);
}

// asked for at once, as in tile_source
__device__ __forceinline__ void ask_for(StateView& sv)
{
    asm volatile("" : "+s"(sv.overflow), "+s"(sv.cur_scale), "+s"(sv.b1t_next), "+s"(sv.b2t_next), "+s"(sv.b1t_rest), "+s"(sv.b2t_rest));
}

template <int ARITH, int WD, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_chunks_gated_kernel(ChunkBatch b, size_t chunk_numel, GatedArgs ga, FirstCall fc,
                             const ps_step_state* __restrict__ st)
{
    const TileSource t = tile_source(b.c[blockIdx.y], b.n[blockIdx.y]);
    const CallSpan s = call_span(fc, blockIdx.x);
    StateView sv = view_state(st);
    ask_for(sv);
    gated_tile<ARITH, WD, NT>(t, blockIdx.x, s, chunk_numel, ga, fc, sv);
}

// The same over evenly spaced chunks.
template <int ARITH, int WD, bool NT>
__device__ __forceinline__ void even_gated_tile(const EvenChunk& t, uint32_t tile, size_t chunk_numel, const GatedArgs& ga, const FirstCall& fc,
                                                const StateView& sv)
{
    const size_t base = (size_t)tile * kTile;
    if (__builtin_expect(sv.overflow, 0)) {
        if (restore_leader(tile)) restore_tiles<NT>(t.p32, t.h16, base, t.numel);
        return;
    }
    if (tile < whole_tiles(t.numel)) {
        LaneTile r;
        tile_load<false, NT>(r, t.p32, t.m32, t.v32, t.h16, base);
        __builtin_amdgcn_sched_barrier(0);
        const CallSpan s = call_span(fc, tile);
        if (!s.cut) {
            const StepConsts c = gated_consts<ARITH>(ga, sv, s.here);
            tile_finish<ARITH, WD, UNSCALE_RUNTIME, false, NT>(c, s.inside ? c.first_step_size : c.step_size, s.inside ? c.first_bc2inv : c.bc2inv,
                                                    r, t.p32, t.m32, t.v32, t.h16, base);
            return;
        }
    }
    const bool here = fc.chunk == (int)blockIdx.y;
    const StepConsts c = gated_consts<ARITH>(ga, sv, here);
    size_t end = t.numel;  // as in gated_tile: zeros behind it that are no fixed point are computed
    if (base + kTile > end && end < chunk_numel && !zeros_are_a_fixed_point(c)) end = chunk_numel;
    if (base >= end) return;
    adam_tile_scalar<ARITH, WD, UNSCALE_RUNTIME>(c, t.p32, t.m32, t.v32, t.h16, base, base + kTile < end ? base + kTile : end,
                                                 here ? fc.lo : 0, here ? fc.hi : 0);
}

template <int ARITH, int WD, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_even_chunks_gated_kernel(float* p32, float* m32, float* v32, uint16_t* h16, uint32_t stride, uint32_t numel, uint32_t last,
                                  uint32_t short_by, const ps_step_state* __restrict__ st, size_t chunk_numel, GatedArgs ga, FirstCall fc)
{
    const EvenChunk t = even_chunk(p32, m32, v32, h16, stride, numel, last, short_by);
    StateView sv = view_state(st);
    ask_for(sv);
    even_gated_tile<ARITH, WD, NT>(t, blockIdx.x, chunk_numel, ga, fc, sv);
}

// ------------------------------------------------------- tensor-list kernels
//
// The same tiles over a list of TENSORS of different lengths, for chunk layouts in which a
// parameter's momentum and variance do not sit at the parameter's own offset (the reference packs
// optimizer-state tensors first-fit in parameters() order, patrickstar/core/client.py:282-309, so the
// whole-chunk pass does not apply and the reference loops over tensors, fp16_cpu_adam.py:336-468).
//
// Grid: x = tile inside a tensor, y = tensor inside the batch, exactly like the chunk-list kernels, so that a
// wave reaches its first data load after ONE scalar load of its descriptor.  The host sorts the tensors by length
// and puts tensors of (nearly) the same length into one launch; x runs up to the longest tensor of the batch and
// the few workgroups beyond a shorter tensor's end leave at once.  (A one-dimensional grid over all tiles with a
// tile -> tensor table costs a second dependent scalar load per wave: 4 to 10 % at this kernel's operating point.)
//
// Tensors start at arbitrary element offsets of their chunks.  The tile grid of a tensor is laid over the ADDRESSES
// of its fp32 parameter, not over its element numbers: the up to 255 elements in front of the parameter's first
// 1 KiB boundary form a tile of their own (done element by element), and every later tile is one whole aligned KiB
// of the fp32 parameter (and of every other list that shares the parameter's phase: the fp16 list does in the
// reference's layout).  Wave accesses at a 256-, 512- or 768-byte phase of a KiB measured 6 to 8 % slower than
// aligned ones (all four lists shifted), 2 % with only the fp16 list at a 256-byte phase.  Momentum and variance
// tensors may sit at ANY element phase against their parameter: their 16-byte accesses then go to addresses that are
// only 4-byte aligned (which the hardware serves: 5.7-5.9 TB/s against 6.1 aligned and 3.7 element by element).

constexpr int kTensorBatch = 64;
struct TensorBatch {
    ps_chunk t[kTensorBatch];          // fp32 param, exp_avg, exp_avg_sq, fp16 slot: addresses of the tile grid's origin
    uint64_t lengths[kTensorBatch];    // low 40 bits: elements from the origin on; high 8 bits: elements in front of it
                                       // (0..255; they are tile 0 of the tensor if there are any); between them: which
                                       // of the launch's constants the tensor takes (steps whose tensors have their own)
    int first_call;                    // which tensor of the batch is the step's first operator call; -1: none
};
constexpr uint64_t kNumelMask = (1ull << 40) - 1;

// One tensor of a launch as its workgroups see it.  Descriptor and lengths are asked for at once (tile_source) instead of
// one after the other: four launches over the upper half of a BERT-base-sized module 216.8 -> 212.6 us, five over all of
// it with a rate per layer 607 -> 604.5 us.
struct TensorView {
    TileSource t;
    size_t numel;
    int head, cls;
    bool first;      // the tensor is the step's first operator call
    uint32_t x;      // this workgroup's number among those of its tensor
    ptrdiff_t tile;  // this workgroup's; -1: the elements in front of the tile grid
};
__device__ __forceinline__ TensorView tensor_view(const TensorBatch& b)
{
    TensorView w;
    w.t = tile_source(b.t[blockIdx.y], b.lengths[blockIdx.y]);
    w.numel = w.t.numel & kNumelMask;
    w.cls = (int)((w.t.numel >> 40) & 0xFFFFu);
    w.head = (int)(w.t.numel >> 56);
    w.first = (int)blockIdx.y == b.first_call;
    w.x = blockIdx.x;
    w.tile = (ptrdiff_t)w.x - (w.head ? 1 : 0);
    return w;
}

// Tensors that lie at the same place of their four lists (the layout that PatrickStarClient makes: momentum and variance
// mirror the parameters' chunks, and so do the lists' allocations): what differs from tensor to tensor is one offset and one
// length, 12 bytes, and one launch takes up to 208 of them, in up to 8 groups of nearly the same length (host-decided, with
// numbers of their own: of up to 24 classes).
//
// The grid is one-dimensional.  Its workgroups are divided among up to 8 segments, tensors of nearly the same length
// each; inside a segment the tensor is a division by the segment's width away (a multiplication by its reciprocal).  A wave
// reaches its first data load after three rounds of scalar loads (segments, segment, tensor) and some 50 scalar
// instructions, where TensorBatch needs one round, so 11 workgroups per CU instead of 9 keep as many loads in flight.
//
// What that buys is the ends of launches, 4 to 9 us each.  Device time in several launches (TensorBatch) / in one, us, lists
// from 28 Mi elements on with the non-temporal hint, where 13 workgroups per CU are resident: BERT-base, 199
// tensors, 463.8 / 459.2 host-decided, 474.7 / 461.0 device-decided with a rate per layer; its upper half, 100 tensors 185.2 / 181.3
// and 192.0 / 184.5; 12 layers of hidden size 64 12.9 / 5.1 and 17.6 / 8.6; 11 M elements with no two tensors at the same phase
// 52.6 / 39.6.  (With plain accesses BERT-base took 517 / 500, under a cap of 9 508, of 12 533.)  Longer lists gain less than
// the longer way to the first load costs them: 335 M elements 1408 / 1423 host-decided, 1426 / 1416 device-decided, 1557 M (GPT-2 XL,
// 580 tensors, three launches) 6568 / 6629 and 6640 / 6612, so lists of more than 256 Mi elements keep TensorBatch.
constexpr int kNearBatch = 208;
constexpr int kSegments = 8;
struct Segment {
    uint32_t start, first;  // workgroup and tensor it begins with
    uint32_t width, magic;  // workgroups per tensor (2 at least); 2^32 / width, rounded up
};
struct NearBatch {
    uint32_t start[kSegments];      // of the second segment, the third ...; behind the last one: 0xFFFFFFFF
    Segment seg[kSegments];
    ps_chunk lists;                 // where offset 0 lies in the four lists
    uint64_t at[kNearBatch];        // low 40 bits: offset of the tile grid's origin; then class and head as in TensorBatch::lengths
    uint32_t numel[kNearBatch];     // elements from the origin on
    int first_call;
};
__device__ __forceinline__ TensorView tensor_view(const NearBatch& b, uint32_t wg)
{
    uint32_t k = 0;
#pragma unroll
    for (int j = 0; j < kSegments - 1; ++j)  // k += wg >= start[j]
        asm("s_cmp_ge_u32 %1, %2\n\ts_addc_u32 %0, %0, 0" : "+s"(k) : "s"(wg), "s"(b.start[j]) : "scc");
    Segment s = b.seg[k];
    float *p32 = b.lists.param_fp32, *m32 = b.lists.exp_avg, *v32 = b.lists.exp_avg_sq;
    uint16_t* h16 = b.lists.param_fp16;
    int first_call = b.first_call;
    asm volatile("" : "+s"(s.start), "+s"(s.first), "+s"(s.width), "+s"(s.magic), "+s"(p32), "+s"(m32), "+s"(v32), "+s"(h16), "+s"(first_call));
    const uint32_t r = wg - s.start;
    uint32_t q = __umulhi(r, s.magic);  // r / width, or one more: then the remainder is negative
    if ((int32_t)(r - q * s.width) < 0) q -= 1;
    const uint32_t index = s.first + q;
    uint64_t at = b.at[index];
    uint32_t numel = b.numel[index];
    asm volatile("" : "+s"(at), "+s"(numel));
    const uint64_t off = at & kNumelMask;
    const uint32_t hi = (uint32_t)(at >> 32);
    TensorView w;
    w.first = (int)index == first_call;
    w.numel = numel;
    w.t = TileSource{p32 + off, m32 + off, v32 + off, h16 + off, numel};
    w.cls = (int)((hi >> 8) & 0xFFFFu);
    w.head = (int)(hi >> 24);
    w.x = r - q * s.width;
    w.tile = (int32_t)w.x - (w.head != 0);
    return w;
}

__device__ __forceinline__ TensorView tensor_view(const NearBatch& b) { return tensor_view(b, blockIdx.x); }

// The elements in front of a tensor's tile grid: indices -head .. -1 relative to the descriptor's addresses.
template <int ARITH, int WD, int UNS>
__device__ __forceinline__ void adam_head(const StepConsts& c, const ps_chunk& t, int head, bool first_call)
{
    const float step_size = first_call ? c.first_step_size : c.step_size;
    const float bc2inv = first_call ? c.first_bc2inv : c.bc2inv;
    for (int j = threadIdx.x; j < head; j += kBlock) {
        const ptrdiff_t i = (ptrdiff_t)j - head;
        float g = half_bits_to_float(t.param_fp16[i]);
        float p = t.param_fp32[i], m = t.exp_avg[i], v = t.exp_avg_sq[i];
        element_any<ARITH, WD, UNS>(c, step_size, bc2inv, g, p, m, v);
        t.param_fp32[i] = p;
        t.exp_avg[i] = m;
        t.exp_avg_sq[i] = v;
        t.param_fp16[i] = (uint16_t)float_to_half_bits(p);
    }
}

// One tile of a tensor, which is one operator call: all of its elements take the first call's scalars, or none.  As in
// adam_tile_late_consts the constants are formed after the tile's loads have been issued.
template <int ARITH, int WD, int UNS, bool NT, typename MakeConsts>
__device__ __forceinline__ void adam_tensor_tile(MakeConsts make_consts, const TensorView& w, bool first)
{
    const ps_chunk t = as_chunk(w.t);
    const size_t base = (size_t)w.tile * kTile;
    const int access = (uint32_t)w.tile < whole_tiles(w.numel) ? tile_access(t) : TILE_ELEMENTWISE;
    if (access == TILE_ALIGNED) {
        LaneTile r;
        tile_load<false, NT>(r, t.param_fp32, t.exp_avg, t.exp_avg_sq, t.param_fp16, base);
        const StepConsts c = make_consts();
        tile_finish<ARITH, WD, UNS, false, NT>(c, first ? c.first_step_size : c.step_size, first ? c.first_bc2inv : c.bc2inv, r, t.param_fp32,
                                    t.exp_avg, t.exp_avg_sq, t.param_fp16, base);
        return;
    }
    if constexpr (!NT) {  // (tensors that stream past the caches have whole lines)
        if (access == TILE_STATE_DWORD_ALIGNED) {
            LaneTile r;
            tile_load<true>(r, t.param_fp32, t.exp_avg, t.exp_avg_sq, t.param_fp16, base);
            const StepConsts c = make_consts();
            tile_finish<ARITH, WD, UNS, true>(c, first ? c.first_step_size : c.step_size, first ? c.first_bc2inv : c.bc2inv, r,
                                              t.param_fp32, t.exp_avg, t.exp_avg_sq, t.param_fp16, base);
            return;
        }
    }
    if (base < w.numel) {  // (the grid is as wide as the longest tensor of the batch)
        const StepConsts c = make_consts();
        const size_t end = base + kTile < w.numel ? base + kTile : w.numel;
        adam_tile_scalar<ARITH, WD, UNS>(c, t.param_fp32, t.exp_avg, t.exp_avg_sq, t.param_fp16, base, end, 0, first ? w.numel : 0);
    }
}

// fp16 <- RNE(fp32) of this workgroup's tiles (a skipped step).
template <bool NT>
__device__ __forceinline__ void restore_tensor_tiles(const ps_chunk& t, const TensorView& w)
{
    if (!restore_leader(w.x)) return;
    if (w.tile >= 0) {
        restore_tiles<NT>(t.param_fp32, t.param_fp16, (size_t)w.tile * kTile, w.numel);
        return;
    }
    // workgroup 0 of a tensor with elements in front of its tile grid: those, and the tiles it leads
    restore_tile(t.param_fp32 - w.head, t.param_fp16 - w.head, 0, (size_t)w.head);
#pragma unroll 1
    for (unsigned u = 1; u < kRestoreTiles; ++u) restore_tile(t.param_fp32, t.param_fp16, (size_t)(u * kRestoreStride - 1) * kTile, w.numel);
}

template <typename LIST, int ARITH, int WD, int UNS, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_kernel(LIST b, StepConsts c)
{
    const TensorView w = tensor_view(b);
    const bool first = w.first;  // a tensor is one operator call: all of its tiles, or none
    if (w.tile < 0) {
        adam_head<ARITH, WD, UNS>(c, as_chunk(w.t), w.head, first);
        return;
    }
    adam_tensor_tile<ARITH, WD, UNS, NT>([&]() { return c; }, w, first);
}

template <typename LIST, int ARITH, int WD, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_gated_kernel(LIST b, GatedArgs ga, const ps_step_state* __restrict__ st)
{
    const TensorView w = tensor_view(b);
    const ps_chunk t = as_chunk(w.t);
    const bool first = w.first;
    const size_t base = w.tile < 0 ? 0 : (size_t)w.tile * kTile;
    if (w.tile >= 0 && base >= w.numel) return;
    const StateView sv = view_state(st);
    if (__builtin_expect(sv.overflow, 0)) {
        restore_tensor_tiles<NT>(t, w);
        return;
    }
    if (w.tile < 0) {
        adam_head<ARITH, WD, UNSCALE_RUNTIME>(gated_consts<ARITH>(ga, sv, first), t, w.head, first);
        return;
    }
    adam_tensor_tile<ARITH, WD, UNSCALE_RUNTIME, NT>([&]() { return gated_consts<ARITH>(ga, sv, first); }, w, first);
}

// A step whose tensors carry their own step numbers and hyper-parameters: calls that come out with the same constants
// form a class.  One launch takes tensors of ANY class (the launch shape depends on the tensors' lengths only, so a
// list in which every tensor is a class of its own runs like a list with one class); TensorBatch::lengths says which
// record of the launch's constants each tensor of the batch uses.  What a launch cannot mix is what the kernels are
// compiled for: the arithmetic, the weight-decay form and the way of unscaling.
// Host-decided: the constants of up to kLaunchClasses classes travel with the launch (a launch's arguments stay
// under 4 KiB: 2696 bytes of NearBatch, which is the larger of the two lists, and 24 x 56 of constants make 4040).
constexpr int kLaunchClasses = 24;
struct ConstsBatch {
    StepConsts c[kLaunchClasses];
};
static_assert(sizeof(TensorBatch) + sizeof(ConstsBatch) <= 4096 && sizeof(NearBatch) + sizeof(ConstsBatch) <= 4096, "kernel arguments of one launch");

// No tensor is "the first call" here: a first call that differs is a class of its own.
template <typename LIST, int ARITH, int WD, int UNS, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_each_kernel(LIST b, ConstsBatch cb)
{
    const TensorView w = tensor_view(b);
    const ps_chunk t = as_chunk(w.t);
    if (w.tile < 0) {
        adam_head<ARITH, WD, UNS>(cb.c[w.cls], t, w.head, false);
        return;
    }
    adam_tensor_tile<ARITH, WD, UNS, NT>([&]() { return cb.c[w.cls]; }, w, false);
}

// The same for tensors whose gradient is binary32 and which have no binary16 copy (PS_TENSOR_GRAD_F32): the
// descriptor's param_fp16 field holds the gradient's address.  Their tile grid starts at the tensor's first element.
template <int ARITH, int WD, int UNS>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_each_f32grad_kernel(TensorBatch b, ConstsBatch cb)
{
    const TensorView w = tensor_view(b);
    const size_t base = (size_t)blockIdx.x * kTile;
    if (base >= w.numel) return;
    adam_tile_f32grad<ARITH, WD, UNS>([&]() { return cb.c[w.cls]; }, w.t.p32, w.t.m32, w.t.v32,
                                      reinterpret_cast<const float*>(w.t.h16), base, w.numel);
}

// Device-decided: the constants of every class are formed on the device by plan_consts_kernel (below), one record
// per class in the caller's workspace, before the update kernels run.
struct PlannedConsts {
    StepConsts c;
    float beta1_t, beta2_t;  // the operator object's beta^t after this call (unused by the torch formula)
};
static_assert(sizeof(PlannedConsts) == 64, "one 64-byte record per class in the caller's workspace");

template <int ARITH, int WD, bool NT, typename Flagged>
__device__ __forceinline__ void planned_tensor(const TensorView& w, const PlannedConsts* __restrict__ consts, Flagged flagged)
{
    const ps_chunk t = as_chunk(w.t);
    const size_t base = w.tile < 0 ? 0 : (size_t)w.tile * kTile;
    if (w.tile >= 0 && base >= w.numel) return;
    if (__builtin_expect(flagged(), 0)) {
        restore_tensor_tiles<NT>(t, w);
        return;
    }
    if (w.tile < 0) {
        adam_head<ARITH, WD, UNSCALE_RUNTIME>(consts[w.cls].c, t, w.head, false);
        return;
    }
    adam_tensor_tile<ARITH, WD, UNSCALE_RUNTIME, NT>(
        [&]() {
            __builtin_amdgcn_sched_barrier(0);  // all of the tile's loads in front of the first wait: with the torch
            // formula the compiler waited behind the third of four, 109 M elements 516 -> 496 us, 223 M 1052 -> 1009
            return consts[w.cls].c;
        },
        w, false);
}

template <typename LIST, int ARITH, int WD, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_planned_kernel(LIST b, const PlannedConsts* __restrict__ consts,
                                const ps_step_state* __restrict__ st)
{
    planned_tensor<ARITH, WD, NT>(tensor_view(b), consts, [&]() { return st->overflow != 0; });
}

// PS_TENSOR_GRAD_F32 tensors of a device-decided step: a flagged step leaves them alone (there is no fp16 copy to
// restore).
template <int ARITH, int WD>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_planned_f32grad_kernel(TensorBatch b, const PlannedConsts* __restrict__ consts,
                                        const ps_step_state* __restrict__ st)
{
    const TensorView w = tensor_view(b);
    const size_t base = (size_t)blockIdx.x * kTile;
    if (base >= w.numel || st->overflow) return;
    adam_tile_f32grad<ARITH, WD, UNSCALE_RUNTIME>([&]() { return consts[w.cls].c; }, w.t.p32, w.t.m32, w.t.v32,
                                                  reinterpret_cast<const float*>(w.t.h16), base, w.numel);
}

__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    restore_chunks_kernel(ChunkBatch b, const ps_step_state* __restrict__ st)
{
    if (st != nullptr && !st->overflow) return;
    const ps_chunk& ch = b.c[blockIdx.y];
    restore_tile(ch.param_fp32, ch.param_fp16, (size_t)blockIdx.x * kTile, b.n[blockIdx.y]);
}

struct CastArgs {
    const float* src;
    uint16_t* dst;
    size_t numel, n_tiles;
};
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    cast_kernel(CastArgs a)
{
    for (size_t t = blockIdx.x; t < a.n_tiles; t += gridDim.x)
        restore_tile(a.src, a.dst, t * (size_t)kTile, a.numel);
}

// ------------------------------------------------- auxiliary (non-hot) kernels

constexpr int kAuxBlock = 256;

// Flat tensor, any grad dtype, optional fp16 output (adam_update of the operator).
// Element-wise accesses: tensors handed to the operator are views at arbitrary
// element offsets inside a chunk, so no alignment can be assumed.
template <int WD, bool GRAD_HALF>
__global__ void __launch_bounds__(kAuxBlock)
    adam_flat_kernel(StepConsts c, float* p32, const void* grads, float* m32, float* v32,
                     uint16_t* out16, size_t numel)
{
    const uint16_t* gh = static_cast<const uint16_t*>(grads);
    const float* gf = static_cast<const float*>(grads);
    size_t stride = (size_t)gridDim.x * kAuxBlock;
    for (size_t i = (size_t)blockIdx.x * kAuxBlock + threadIdx.x; i < numel; i += stride) {
        float g = GRAD_HALF ? half_bits_to_float(gh[i]) : gf[i];
        float p = p32[i], m = m32[i], v = v32[i];
        element_any<PS_ARITH_OPERATOR, WD, UNSCALE_RUNTIME>(c, c.step_size, c.bc2inv, g, p, m, v);
        p32[i] = p;
        m32[i] = m;
        v32[i] = v;
        if (out16) out16[i] = (uint16_t)float_to_half_bits(p);
    }
}

// The same operator with vector accesses: single-wave workgroups over 256-element tiles, one tile per workgroup, the
// resident-workgroup cap and the order "all loads, arithmetic, all stores" of the chunk-list kernels, every variant
// (weight-decay form, unscale form, gradient type, fp16 output or none) a compile-time property so that a wave runs
// straight through.  The tile grid is laid over the ADDRESSES of the fp32 parameter: the pointers are those of the
// parameter's first 1 KiB boundary, so every wave access covers one aligned KiB (tiles at another phase of a KiB
// measured 6 to 8 % slower); the up to 255 elements in front of it (`head`) and the up to 255 behind the last whole
// tile (`tail`), if there are any, are done element-wise by one extra workgroup of the same launch.  Gradients are read
// only and must share the parameter's 16-byte phase, as must the optional fp16 output.
//
// Addresses and lengths come first so that they are preloaded into scalar registers (-amdgpu-kernarg-preload-count): a
// wave issues its data loads without waiting for its arguments, and the constants are loaded in their shadow.  Of a tensor
// that is a launch of its own that is most of what is left beside the 1.7 us of an empty launch and the bytes: 147 K elements
// 2.52 -> 2.31 us, 590 K 5.03 -> 4.55, 2.36 M 13.35 -> 13.0; from 4096 to 40 K 1.9 -> 2.0.  Kernels of short or lone
// launches, which the preloading makes 0.1 to 0.25 us longer (the element-wise operator, the lone gradient copy, the cast), take
// their arguments in a struct, which is not preloaded.
// STATE_DWORD_ALIGNED: exp_avg / exp_avg_sq sit at another 16-byte phase than the parameter (any element offset).
template <int WD, int UNS, bool GRAD_HALF, bool HAS_OUT, bool STATE_DWORD_ALIGNED, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_flat_vec_kernel(float* p32, const void* grads, float* m32, float* v32,
                         uint16_t* out16,  // may alias grads (fp16 gradients overwritten by fp16 parameters)
                         uint32_t n_tiles, int head, int tail, StepConsts c)
{
    static_assert(kBlock == 64 && kLaneElems == 4 && kUnroll == 1, "one wave, one 16-byte access per lane and fp32 array");
    const size_t t = blockIdx.x;
    if (blockIdx.x == n_tiles) {
        for (int j = threadIdx.x; j < head + tail; j += kBlock) {
            const ptrdiff_t i = j < head ? (ptrdiff_t)j - head : (ptrdiff_t)((size_t)n_tiles * kTile) + (j - head);
            float g = GRAD_HALF ? half_bits_to_float(static_cast<const uint16_t*>(grads)[i])
                                : static_cast<const float*>(grads)[i];
            float p = p32[i], m = m32[i], v = v32[i];
            adam_element<PS_ARITH_OPERATOR, WD, UNS>(c, c.step_size, c.bc2inv, g, p, m, v);
            p32[i] = p;
            m32[i] = m;
            v32[i] = v;
            if (HAS_OUT) out16[i] = (uint16_t)float_to_half_bits(p);
        }
        return;
    }
    const size_t i = (t * kBlock + threadIdx.x) * 4;
    uint2v w;
    float4v gv;
    if (GRAD_HALF)
        w = NT ? __builtin_nontemporal_load((const guint2v*)(static_cast<const uint16_t*>(grads) + i)) : *(const guint2v*)(static_cast<const uint16_t*>(grads) + i);
    else
        gv = ld_f4<NT>(static_cast<const float*>(grads) + i);
    float4v p = ld_f4<NT>(p32 + i), m = ld_f4_as<STATE_DWORD_ALIGNED, NT>(m32 + i), v = ld_f4_as<STATE_DWORD_ALIGNED, NT>(v32 + i);
    float g[4];
    if (GRAD_HALF) {
        g[0] = half_bits_to_float(w[0] & 0xFFFFu);
        g[1] = half_bits_to_float(w[0] >> 16);
        g[2] = half_bits_to_float(w[1] & 0xFFFFu);
        g[3] = half_bits_to_float(w[1] >> 16);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] = gv[e];
    }
    uint32_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float pe = p[e], me = m[e], ve = v[e];
        adam_element<PS_ARITH_OPERATOR, WD, UNS>(c, c.step_size, c.bc2inv, g[e], pe, me, ve);
        p[e] = pe;
        m[e] = me;
        v[e] = ve;
        h[e] = float_to_half_bits(pe);
    }
    st_f4<NT>(p32 + i, p);
    st_f4_as<STATE_DWORD_ALIGNED, NT>(m32 + i, m);
    st_f4_as<STATE_DWORD_ALIGNED, NT>(v32 + i, v);
    if (HAS_OUT) {
        uint2v o;
        o[0] = h[0] | (h[1] << 16);
        o[1] = h[2] | (h[3] << 16);
        if (NT)
            __builtin_nontemporal_store(o, (guint2v*)(out16 + i));
        else
            *(guint2v*)(out16 + i) = o;
    }
}

// ----------------------------------------------------------- overflow scan
//
// A binary16 value is inf or nan iff its five exponent bits are all set.
// For a 32-bit word holding two halves: mask the exponents, add one unit of
// the lowest exponent bit to each; an all-ones exponent carries into bit 15 /
// bit 31 (the masked low half is at most 0x7C00, so its carry stops at bit 15).

__device__ __forceinline__ uint32_t nonfinite_halves(uint32_t w)
{
    return ((w & 0x7C007C00u) + 0x04000400u) & 0x80008000u;
}
// A binary32 value is inf or nan iff its eight exponent bits are all set.
__device__ __forceinline__ uint32_t nonfinite_float(uint32_t w) { return ((w & 0x7F800000u) == 0x7F800000u) ? 1u : 0u; }

// OR across the block: shuffle butterfly inside each wave, LDS across the
// waves of the block (if it has several), then at most one atomic per block (none when nothing was seen).
template <int BLOCK = kAuxBlock>
__device__ __forceinline__ void block_flag_commit(uint32_t hit, uint32_t* flag)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) hit |= (uint32_t)__shfl_xor((int)hit, off, 64);
    if (BLOCK == 64) {
        if (threadIdx.x == 0 && hit) atomicOr(flag, 1u);
        return;
    }
    __shared__ uint32_t wave_hit[BLOCK / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wave_hit[wave] = hit;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t any = 0;
#pragma unroll
        for (int w = 0; w < BLOCK / 64; ++w) any |= wave_hit[w];
        if (any) atomicOr(flag, 1u);
    }
}

// Launch shape of the probe kernels that commit to the device flag: threads per workgroup, 16-byte loads per lane,
// and an unused dynamic-LDS request that caps the resident workgroups per CU (0: no cap).
constexpr int kScanBlock = PS_SCAN_BLOCK;
constexpr int kScanUnroll = PS_SCAN_UNROLL;
constexpr int kScanTile = kScanBlock * 8 * kScanUnroll;  // halves per tile
constexpr size_t kScanLdsBytes = (size_t)PS_SCAN_LDS_KB * 1024;
// The two-stage probe keeps one partial word per tile: tiles twice as large, so that the word array stays small, in
// the same single-wave launch shape (probe + reduction over 3.2 GB: 0.490 ms, against 0.512 ms with 256-thread
// workgroups without a cap).
constexpr int kPartialBlock = 64;
constexpr int kPartialUnroll = 16;
constexpr int kPartialTile = kPartialBlock * 8 * kPartialUnroll;  // 8192 halves = 16 KiB per tile

// 16 bytes at an address that is only aligned to the element (the hardware serves multi-dword global loads at any
// byte address).
typedef uint4v __attribute__((aligned(2))) uint4v_half_aligned;
typedef uint4v __attribute__((aligned(4))) uint4v_word_aligned;

// One scan tile of a buffer of binary16 or binary32 bit patterns, by a workgroup of BLOCK threads: UNROLL 16-byte loads
// per lane, all of them in flight before the first is looked at.  A tile that the buffer ends in, or a buffer that does
// not start on a 16-byte boundary, takes the same number of loads: lanes behind the last whole vector read that vector
// again (it is inside the buffer, and an OR does not mind), the up to 7 (3) elements behind it go one to a lane.
// As a loop over single elements such a tile was a chain of up to 64 waits for memory, and the launch was no faster
// than that chain: 12.2 us for 3 chunks of 6267 halves (2.8 us now), 70.1 us for the four part-filled chunks of a
// BERT-base-sized module (62.6 us now; 109 M halves, read while the update before it is still being written back).
template <typename Element, int BLOCK, int UNROLL, bool NT = false>
__device__ __forceinline__ uint32_t scan_tile(const Element* __restrict__ x, size_t numel, size_t tile)
{
    constexpr bool kHalf = sizeof(Element) == 2;
    constexpr unsigned kVec = 16 / sizeof(Element);  // elements per load
    constexpr size_t kElems = (size_t)BLOCK * kVec * UNROLL;
    typedef typename std::conditional<kHalf, uint4v_half_aligned, uint4v_word_aligned>::type loose_vec;
    auto nonfinite = [](const uint4v& w) {
        uint32_t hit = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) hit |= kHalf ? nonfinite_halves(w[k]) : nonfinite_float(w[k]);
        return hit;
    };
    const size_t base = tile * kElems;
    if (base >= numel) return 0;
    const size_t left = numel - base;
    const Element* t = x + base;
    uint32_t hit = 0;
    uint4v w[UNROLL];
    if ((((uintptr_t)x) & 15u) == 0 && left >= kElems) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
            w[u] = ld_u4<NT>(reinterpret_cast<const uint16_t*>(t + (size_t)(u * BLOCK + threadIdx.x) * kVec));
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) hit |= nonfinite(w[u]);
        return hit;
    }
    const unsigned here = (unsigned)(left < kElems ? left : kElems);
    const unsigned n_vec = here / kVec;
    const unsigned behind = n_vec * kVec + threadIdx.x;
    const uint32_t odd = *(const PS_GLOBAL Element*)(t + (behind < here ? behind : here - 1));
    if (n_vec != 0) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const unsigned i = u * BLOCK + threadIdx.x;
            w[u] = *(const PS_GLOBAL loose_vec*)(t + (size_t)(i < n_vec ? i : n_vec - 1) * kVec);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) hit |= nonfinite(w[u]);
    }
    return hit | (kHalf ? nonfinite_halves(odd) : nonfinite_float(odd));
}

__global__ void __launch_bounds__(kScanBlock)
    scan_f16_kernel(const uint16_t* __restrict__ h, size_t numel, size_t n_tiles,
                    ps_step_state* st)
{
    uint32_t hit = 0;
    for (size_t t = blockIdx.x; t < n_tiles; t += gridDim.x) hit |= scan_tile<uint16_t, kScanBlock, kScanUnroll>(h, numel, t);
    block_flag_commit<kScanBlock>(hit, &st->overflow);
}

constexpr int kScanTileF32 = kScanBlock * 4 * kScanUnroll;  // floats per tile of the binary32 probe

__global__ void __launch_bounds__(kScanBlock)
    scan_f32_kernel(const float* __restrict__ f, size_t numel, size_t n_tiles, ps_step_state* st)
{
    const uint32_t* w = reinterpret_cast<const uint32_t*>(f);
    uint32_t hit = 0;
    for (size_t t = blockIdx.x; t < n_tiles; t += gridDim.x) hit |= scan_tile<uint32_t, kScanBlock, kScanUnroll>(w, numel, t);
    block_flag_commit<kScanBlock>(hit, &st->overflow);
}

// The probe's part of one workgroup, `width` tiles a chunk.  STREAMS: beyond the first `keep` tiles of the list past the caches
// (kScanKeepElements).
template <bool STREAMS>
__device__ __forceinline__ uint32_t probe_tile(const uint16_t* h, size_t n, uint32_t tile, uint32_t width, uint32_t keep)
{
    if (STREAMS && blockIdx.y * width + tile >= keep) return scan_tile<uint16_t, kScanBlock, kScanUnroll, true>(h, n, tile);
    return scan_tile<uint16_t, kScanBlock, kScanUnroll, false>(h, n, tile);
}

template <bool STREAMS>
__global__ void __launch_bounds__(kScanBlock)
    scan_chunks_kernel(ChunkBatch b, ps_step_state* st, uint32_t keep)
{
    uint32_t hit = probe_tile<STREAMS>(b.c[blockIdx.y].param_fp16, b.n[blockIdx.y], blockIdx.x, gridDim.x, keep);
    block_flag_commit<kScanBlock>(hit, &st->overflow);
}

template <bool STREAMS>
__global__ void __launch_bounds__(kScanBlock)
    scan_even_chunks_kernel(const uint16_t* h16, uint32_t stride, uint32_t numel, uint32_t last, uint32_t short_by, ps_step_state* st, uint32_t keep)
{
    const uint32_t n = numel - (blockIdx.y == last ? short_by : 0u);
    uint32_t hit = probe_tile<STREAMS>(h16 + (size_t)stride * blockIdx.y, n, blockIdx.x, gridDim.x, keep);
    block_flag_commit<kScanBlock>(hit, &st->overflow);
}

// The same probe without atomics and without a caller-side state: every workgroup leaves the OR over its tile in
// its own word of a partial-result array; a second, small kernel ORs those words into the caller's flag.
__global__ void __launch_bounds__(kPartialBlock)
    scan_chunks_partial_kernel(ChunkBatch b, uint32_t* __restrict__ partial)
{
    static_assert(kPartialBlock == 64, "one wave per workgroup: the shuffle butterfly is the whole reduction");
    uint32_t hit = scan_tile<uint16_t, kPartialBlock, kPartialUnroll>(b.c[blockIdx.y].param_fp16, b.n[blockIdx.y], blockIdx.x);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) hit |= (uint32_t)__shfl_xor((int)hit, off, 64);
    // written unconditionally: the array keeps whatever an earlier call left in it
    if (threadIdx.x == 0) partial[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = hit ? 1u : 0u;
}

constexpr int kReduceBlock = 1024;
__global__ void __launch_bounds__(kReduceBlock)
    scan_reduce_kernel(const uint32_t* __restrict__ partial, size_t n_words, uint32_t* flag)
{
    __shared__ uint32_t wave_hit[kReduceBlock / 64];
    // every workgroup takes one slice of the words; those that find a hit all store the same 1
    const size_t per = (n_words + gridDim.x - 1) / gridDim.x;
    const size_t lo = (size_t)blockIdx.x * per;
    const size_t hi = lo + per < n_words ? lo + per : n_words;
    uint32_t hit = 0;
#pragma unroll 8
    for (size_t i = lo + threadIdx.x; i < hi; i += kReduceBlock) hit |= partial[i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) hit |= (uint32_t)__shfl_xor((int)hit, off, 64);
    if ((threadIdx.x & 63) == 0) wave_hit[threadIdx.x >> 6] = hit;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t any = 0;
#pragma unroll
        for (int w = 0; w < kReduceBlock / 64; ++w) any |= wave_hit[w];
        if (any) *flag = 1u;  // sticky, like ps_step_state::overflow: only ever set here
    }
}

// Backward-side producer: copy gradients into their slots of the fp16 chunks (patrickstar/core/hook.py:212-216) and probe
// them for inf/nan in the same pass (loss_scaler.py:133-155), instead of a separate cast + sum + host sync per
// parameter.  fp32 gradients are rounded to fp16 (RNE); the probe looks at the value that lands in the chunk.
//
// One launch takes up to 64 gradients, one-dimensional grid, kCopySpan elements of one gradient per workgroup: a copy is
// two waits for memory whatever its length, and a model has more small parameters (biases, norms) than large ones.
// Which gradient a workgroup belongs to: lane k of every wave looks at the first workgroup of gradient k, and the
// number of lanes that find it at or below their own workgroup says it (one load and a ballot, no search).
//
// A slot starts at any element of its chunk and sets the grid: one 16-byte store per lane to the slot's 16-byte
// boundaries.  The source is then at any phase; its 16-byte loads only need the element's alignment (the hardware
// serves multi-dword global loads at any byte address).
//
// Bound by memory where it is long: one gradient of 64 Mi elements 38.0 us (fp16), 68.4 us (fp32), with the look-up
// 38.7 and 69.1 us; with the look-up and 2, 4 and 8 vectors per lane 39.4 / 39.6 / 40.0 and 70.1 / 71.6 / 78.0 us.  The
// 199 gradients of a BERT-base-sized module, a kernel for each: 613 us (2.5 us for every bias); in five launches: 80 us.
constexpr int kGradBatch = 64;
constexpr int kCopyBlock = PS_COPY_BLOCK;
constexpr unsigned kCopySpan = kCopyBlock * 8;  // elements per workgroup
struct GradBatch {
    const void* src[kGradBatch];
    uint16_t* dst[kGradBatch];
    uint64_t numel_half[kGradBatch];   // 2 * elements + (1: the gradient is binary16)
    uint32_t first_block[kGradBatch];  // entries behind the last gradient: 0xFFFFFFFF
};
static_assert(kGradBatch == 64, "one lane per gradient");
static_assert(sizeof(GradBatch) <= 2048, "kernel arguments of one launch");

// Elements [lo, hi) of a gradient, one at a time: the at most 7 in front of the slot's first 16-byte boundary and
// behind its last whole vector, and addresses that are not even element-aligned.
template <bool SRC_HALF>
__device__ __forceinline__ uint32_t copy_elements(const void* src, uint16_t* dst, size_t lo, size_t hi)
{
    uint32_t hit = 0;
    for (size_t i = lo + threadIdx.x; i < hi; i += kCopyBlock) {
        uint32_t h = SRC_HALF ? (uint32_t) static_cast<const uint16_t*>(src)[i] : float_to_half_bits(static_cast<const float*>(src)[i]);
        dst[i] = (uint16_t)h;
        hit |= nonfinite_halves(h);
    }
    return hit;
}

// Workgroup `block` of one gradient.
template <bool SRC_HALF>
__device__ __forceinline__ uint32_t copy_span(const void* src, uint16_t* dst, size_t numel, uint32_t block)
{
    constexpr unsigned esz = SRC_HALF ? 2 : 4;
    if (((uintptr_t)dst & 1u) | ((uintptr_t)src & (esz - 1))) {
        const size_t lo = (size_t)block * kCopySpan;
        return copy_elements<SRC_HALF>(src, dst, lo, lo + kCopySpan < numel ? lo + kCopySpan : numel);
    }
    size_t head = ((16 - ((uintptr_t)dst & 15u)) & 15u) / 2;
    if (head > numel) head = numel;
    const size_t n_vec = (numel - head) / 8;
    uint32_t hit = 0;
    const size_t j = (size_t)block * kCopyBlock + threadIdx.x;
    if (j < n_vec) {
        const size_t at = head + 8 * j;
        uint4v o;
        if (SRC_HALF) {
            o = *(const PS_GLOBAL uint4v_half_aligned*)(static_cast<const uint16_t*>(src) + at);
        } else {
            const float4v x = *(const PS_GLOBAL float4v_dword_aligned*)(static_cast<const float*>(src) + at);
            const float4v y = *(const PS_GLOBAL float4v_dword_aligned*)(static_cast<const float*>(src) + at + 4);
            o[0] = float_to_half_bits(x[0]) | (float_to_half_bits(x[1]) << 16);
            o[1] = float_to_half_bits(x[2]) | (float_to_half_bits(x[3]) << 16);
            o[2] = float_to_half_bits(y[0]) | (float_to_half_bits(y[1]) << 16);
            o[3] = float_to_half_bits(y[2]) | (float_to_half_bits(y[3]) << 16);
        }
        hit = nonfinite_halves(o[0]) | nonfinite_halves(o[1]) | nonfinite_halves(o[2]) | nonfinite_halves(o[3]);
        st_u4(dst + at, o);
    }
    if (block == 0) {
        hit |= copy_elements<SRC_HALF>(src, dst, 0, head);
        hit |= copy_elements<SRC_HALF>(src, dst, head + 8 * n_vec, numel);
    }
    return hit;
}

__device__ __forceinline__ void copy_and_probe(const void* src, uint16_t* dst, uint64_t numel_half, uint32_t block, ps_step_state* st)
{
    const uint32_t hit = (numel_half & 1u) ? copy_span<true>(src, dst, numel_half >> 1, block) : copy_span<false>(src, dst, numel_half >> 1, block);
    if (st != nullptr) block_flag_commit<kCopyBlock>(hit, &st->overflow);
}

__global__ void __launch_bounds__(kCopyBlock) grads_to_chunks_kernel(GradBatch b, ps_step_state* st)
{
    const uint64_t begun = __ballot(b.first_block[threadIdx.x & 63] <= blockIdx.x);
    const int k = __builtin_amdgcn_readfirstlane(__popcll(begun) - 1);  // gradient 0 begins at workgroup 0: never -1
    copy_and_probe(b.src[k], b.dst[k], b.numel_half[k], blockIdx.x - b.first_block[k], st);
}

// A gradient that has the launch to itself: nothing to look up, and arguments of 32 bytes instead of 1.8 KiB (with
// those a launch back to back takes 4.5 us instead of 3.9 up to 1 Mi elements, 6.7 instead of 6.0 for 9 Mi in fp16).
struct GradCopy {
    const void* src;
    uint16_t* dst;
    uint64_t numel_half;
    ps_step_state* st;
};
__global__ void __launch_bounds__(kCopyBlock) grad_to_chunk_kernel(GradCopy c)
{
    copy_and_probe(c.src, c.dst, c.numel_half, blockIdx.x, c.st);
}

// ------------------------------------------------ device-resident step state

__global__ void state_init_kernel(ps_step_state* st, ps_step_state init)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *st = init;
}

struct SeedArgs {
    int64_t adam_step;
    float beta1, beta2, b1t_rest, b2t_rest;
    double beta1_f64, beta2_f64, bc1_next, bc2_next;
    int fresh_operator;
};

__global__ void state_seed_kernel(ps_step_state* st, SeedArgs a)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        // IncrementStep (cpu_adam.h:143-162) for the first call of step adam_step + 1: changed betas restart from
        // pow; else the running product continues only if the object's own step is adam_step
        if (a.fresh_operator) {
            // a new native object (cpu_adam.h:68-86), created with these betas: step 0, beta^t = 1
            st->operator_step = 0;
            st->beta1_t_cur = 1.0f;
            st->beta2_t_cur = 1.0f;
            st->operator_beta1 = a.beta1;
            st->operator_beta2 = a.beta2;
        }
        const bool same_betas = st->operator_beta1 == a.beta1 && st->operator_beta2 == a.beta2;
        const bool follows = same_betas && st->operator_step == a.adam_step;
        st->adam_step = a.adam_step;
        st->beta1 = a.beta1;
        st->beta2 = a.beta2;
        st->beta1_t_next = follows ? st->beta1_t_cur * a.beta1 : a.b1t_rest;
        st->beta2_t_next = follows ? st->beta2_t_cur * a.beta2 : a.b2t_rest;
        st->beta1_t_rest = a.b1t_rest;
        st->beta2_t_rest = a.b2t_rest;
        st->beta1_f64 = a.beta1_f64;
        st->beta2_f64 = a.beta2_f64;
        st->bias_correction1_next = a.bc1_next;
        st->bias_correction2_next = a.bc2_next;
    }
}

// beta ** n for a non-negative integer n in binary64, by squaring in double-double arithmetic: the
// result is the correctly rounded power except within ~2^-90 of a rounding boundary, which is what
// Python's float ** int (the C library's pow) returns for all but about one step in 10^4; the
// float constants derived from 1 - beta ** n did not differ on any of 1.8 million (beta, n) pairs.
struct TwoDouble {
    double hi, lo;
};
__device__ inline TwoDouble two_double_mul(TwoDouble a, TwoDouble b)
{
    double p = a.hi * b.hi;
    double e = __builtin_fma(a.hi, b.hi, -p);
    e += a.hi * b.lo + a.lo * b.hi;
    double s = p + e;
    return TwoDouble{s, e - (s - p)};
}
__device__ inline double pow_int(double base, int64_t n)
{
    TwoDouble r{1.0, 0.0}, x{base, 0.0};
    while (n > 0) {
        if (n & 1) r = two_double_mul(r, x);
        n >>= 1;
        if (n) x = two_double_mul(x, x);
    }
    return r.hi;
}

// ------------------------------------- per-tensor step numbers: constants of a device-decided step
//
// One distinct call of the step (ps_adam_step_tensors_each): its hyper-parameters, its distance d from the device's
// step counter, and how Adam_Optimizer::IncrementStep (cpu_adam.h:143-162) treats it, which the host can tell from
// the call before it:
//   PLAN_FIRST  the step's first operator call: continues the object's running product if the object, as the last
//               clean step left it, stands at this call's step minus one with the same betas; else pow
//   PLAN_MUL    its step number is the previous call's plus one, same betas: the previous call's beta^t times beta
//   PLAN_POW    anything else: (float)pow((double)beta, step)
//   PLAN_TORCH  the torch formula: 1 - beta ** step in binary64, no operator call
enum { PLAN_POW = 0, PLAN_FIRST = 1, PLAN_MUL = 2, PLAN_TORCH = 3 };
constexpr int32_t PLAN_KIND_MASK = 0xFF;
constexpr int32_t PLAN_GRAD_F32 = 0x100;  // or-ed into PlanClass::mode: the tensors' gradients are binary32 (the clamp bound differs)
struct PlanClass {
    double lr, beta1, beta2, eps, wd;
    int64_t d;     // the call's step number is adam_step + 1 + d
    int32_t mode;  // one of the kinds above, plus PLAN_GRAD_F32
    int32_t prev;  // PLAN_MUL: the class (index in the table) of the call before it
};
constexpr int kPlanBatch = 64;  // one lane per class; 64 x 56 bytes of kernel arguments
template <int N>
struct PlanBatchOf {
    PlanClass k[N];
};
using PlanBatch = PlanBatchOf<kPlanBatch>;
struct PlanArgs {
    double grad_clamp;
    int64_t last_d;             // of the step's last operator call
    int adamw, bias_correction;
    int first_class, n;         // this launch covers classes [first_class, first_class + n) of the table
    int is_last_launch;         // the launch that leaves the pending record
    int last_operator_class;    // class of the step's last operator call; -1: the step calls the operator for nothing
    float last_beta1, last_beta2;
};

// By one wave.
template <int N>
__device__ __forceinline__ void plan_consts(const PlanBatchOf<N>& pb, const PlanArgs& a, ps_step_state* st, PlannedConsts* table)
{
    __shared__ float b1t_of[N], b2t_of[N];
    const int j = threadIdx.x;
    const int64_t adam_step = st->adam_step;
    const double cur_scale = st->cur_scale;
    const bool bias = a.bias_correction != 0;
    PlanClass k;
    memset(&k, 0, sizeof(k));
    if (j < a.n) k = pb.k[j];
    const int kind = k.mode & PLAN_KIND_MASK;
    uint64_t multiplying = __ballot(kind == PLAN_MUL);
    if (j < a.n && kind != PLAN_MUL) {
        const float clip = clamp_bound(a.grad_clamp, cur_scale, (k.mode & PLAN_GRAD_F32) != 0);
        const int64_t t = adam_step + 1 + k.d;
        PlannedConsts out;
        if (kind == PLAN_TORCH) {
            torch_consts(out.c, k.lr, k.beta1, k.beta2, k.eps, k.wd, a.adamw != 0, bias ? 1.0 - pow_int(k.beta1, t) : 1.0,
                         bias ? 1.0 - pow_int(k.beta2, t) : 1.0, cur_scale, clip);
            out.beta1_t = out.beta2_t = 0.0f;
        } else {
            const float b1 = (float)k.beta1, b2 = (float)k.beta2;
            const bool follows = kind == PLAN_FIRST && st->operator_beta1 == b1 && st->operator_beta2 == b2 &&
                                 st->operator_step + 1 == t;
            out.beta1_t = follows ? st->beta1_t_cur * b1 : (float)pow_int((double)b1, t);
            out.beta2_t = follows ? st->beta2_t_cur * b2 : (float)pow_int((double)b2, t);
            finish_consts(out.c, (float)k.lr, b1, b2, (float)k.eps, (float)k.wd, a.adamw != 0, out.beta1_t, out.beta2_t,
                          bias, (float)cur_scale, clip);
        }
        b1t_of[j] = out.beta1_t;
        b2t_of[j] = out.beta2_t;
        table[a.first_class + j] = out;
    }
    __syncthreads();
    if (j != 0) return;
    // a call that multiplies needs the call before it: in order, by one lane, which looks at those calls only (a look at each
    // of the classes was a chain of waits: 14 classes of which none multiplies cost a step 4.2 us, now 2.7)
    for (; multiplying != 0; multiplying &= multiplying - 1) {
        const int i = (int)__builtin_ctzll(multiplying);
        const PlanClass& k = pb.k[i];
        const float clip = clamp_bound(a.grad_clamp, cur_scale, (k.mode & PLAN_GRAD_F32) != 0);
        const int q = k.prev - a.first_class;  // an earlier class: of this launch, or of a launch before it
        const float p1 = q >= 0 ? b1t_of[q] : table[k.prev].beta1_t;
        const float p2 = q >= 0 ? b2t_of[q] : table[k.prev].beta2_t;
        PlannedConsts out;
        const float b1 = (float)k.beta1, b2 = (float)k.beta2;
        out.beta1_t = p1 * b1;
        out.beta2_t = p2 * b2;
        finish_consts(out.c, (float)k.lr, b1, b2, (float)k.eps, (float)k.wd, a.adamw != 0, out.beta1_t, out.beta2_t, bias,
                      (float)cur_scale, clip);
        b1t_of[i] = out.beta1_t;
        b2t_of[i] = out.beta2_t;
        table[a.first_class + i] = out;
    }
    if (!a.is_last_launch) return;
    if (a.last_operator_class < 0) {
        st->pending_operator_step = 0;
        return;
    }
    const int q = a.last_operator_class - a.first_class;
    st->pending_beta1_t = q >= 0 ? b1t_of[q] : table[a.last_operator_class].beta1_t;
    st->pending_beta2_t = q >= 0 ? b2t_of[q] : table[a.last_operator_class].beta2_t;
    st->pending_beta1 = a.last_beta1;
    st->pending_beta2 = a.last_beta2;
    st->pending_operator_step = adam_step + 1 + a.last_d;
}

__global__ void __launch_bounds__(64)
    plan_consts_kernel(PlanBatch pb, PlanArgs a, ps_step_state* st, PlannedConsts* table)
{
    plan_consts(pb, a, st, table);
}

__global__ void state_set_scaler_kernel(ps_step_state* st, double cur_scale, int scale_is_int,
                                        int64_t cur_iter, int64_t last_overflow_iter,
                                        int cur_hysteresis)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        st->cur_scale = cur_scale;
        st->scale_is_int = scale_is_int;
        st->cur_iter = cur_iter;
        st->last_overflow_iter = last_overflow_iter;
        st->cur_hysteresis = cur_hysteresis;
    }
}

// What DynamicLossScaler.update_scale (loss_scaler.py:158-182) makes of the state, formed by one whole wave (every lane
// the same, except that lanes 0 to 3 raise one beta each; the shuffles that hand the powers round need all 64 of them).
// `operator_calls`: how many times the step that was just queued called the native operator in the reference's terms (its
// tensors; 0 when every chunk took the torch formula): a clean step moves the operator's own step / beta^t state accordingly
// (Adam_Optimizer::IncrementStep, cpu_adam.h:143-162), a skipped step never reaches the operator.
__device__ __forceinline__ ps_step_state scaler_updated(ps_step_state s, bool overflow, int64_t operator_calls)
{
    if (overflow) {
        if (s.delayed_shift == 1 || s.cur_hysteresis == 1) {
            // Python: max(cur_scale / scale_factor, min_scale) -- true division gives a
            // float; max keeps its first argument unless the second is strictly greater.
            double q = s.cur_scale / s.scale_factor;
            if (s.min_scale > q) {
                s.cur_scale = s.min_scale;
                s.scale_is_int = s.min_is_int;
            } else {
                s.cur_scale = q;
                s.scale_is_int = 0;
            }
        } else {
            s.cur_hysteresis -= 1;
        }
        s.last_overflow_iter = s.cur_iter;
        s.skipped_steps += 1;
    } else {
        if (s.consecutive_hysteresis) s.cur_hysteresis = s.delayed_shift;
        if ((s.cur_iter - s.last_overflow_iter) % s.scale_window == 0) {
            if (!s.consecutive_hysteresis) s.cur_hysteresis = s.delayed_shift;
            s.cur_scale = s.cur_scale * s.scale_factor;
            s.scale_is_int = s.scale_is_int && s.factor_is_int;
        }
        // the step ran: state["step"] += 1
        const int64_t t = s.adam_step + 1;
        s.adam_step = t;
        if (s.pending_operator_step != 0) {
            // a step whose tensors carried their own step numbers and betas: what its last call left
            s.operator_step = s.pending_operator_step;
            s.beta1_t_cur = s.pending_beta1_t;
            s.beta2_t_cur = s.pending_beta2_t;
            s.operator_beta1 = s.pending_beta1;
            s.operator_beta2 = s.pending_beta2;
        } else if (operator_calls >= 1) {
            // what the operator object holds after its last call of step t: the first call's beta^t if it
            // was the only one, else pow(beta, t) from the second call on
            s.beta1_t_cur = operator_calls == 1 ? s.beta1_t_next : s.beta1_t_rest;
            s.beta2_t_cur = operator_calls == 1 ? s.beta2_t_next : s.beta2_t_rest;
            s.operator_step = t;
            s.operator_beta1 = s.beta1;
            s.operator_beta2 = s.beta2;
        }
        // step t + 1: every call after the first evaluates (float)pow((double)beta, t + 1); the first call
        // multiplies the held value by beta if the object's step is t, else it evaluates pow as well.  And
        // fp16_cpu_adam.py:412-413 for that step: the powers of the betas that are no floats
        const int j = threadIdx.x & 3;
        const double power = pow_int(j == 0 ? (double)s.beta1 : j == 1 ? (double)s.beta2 : j == 2 ? s.beta1_f64 : s.beta2_f64, t + 1);
        s.beta1_t_rest = (float)__shfl(power, 0, 64);
        s.beta2_t_rest = (float)__shfl(power, 1, 64);
        const bool follows = s.operator_step == t && s.operator_beta1 == s.beta1 && s.operator_beta2 == s.beta2;
        s.beta1_t_next = follows ? s.beta1_t_cur * s.beta1 : s.beta1_t_rest;
        s.beta2_t_next = follows ? s.beta2_t_cur * s.beta2 : s.beta2_t_rest;
        s.bias_correction1_next = 1.0 - __shfl(power, 2, 64);
        s.bias_correction2_next = 1.0 - __shfl(power, 3, 64);
    }
    s.cur_iter += 1;
    s.last_skipped = overflow ? 1u : 0u;
    s.overflow = 0;
    s.pending_operator_step = 0;
    return s;
}

// One lane's work: the state as it now is, and the log's record of the iteration.  Field by field, as far as scaler_updated changes them:
// the reserved arrays of a state that is stored as a whole go through memory (3 KiB of LDS for every workgroup of a kernel that does
// so, 64 KiB and scratch memory in adam_small_step_kernel: 75 tiles 7.0 -> 6.4 us, waited for 18.9 -> 17.6, 240 tiles 7.6 -> 6.5; three launches of 4096 tiles 12.1 -> 10.9).
__device__ __forceinline__ void scaler_store(ps_step_state* st, const ps_step_state& s, ps_scale_record* log, int64_t log_capacity)
{
    if (log != nullptr && log_capacity > 0) {
        ps_scale_record r;
        r.scale_after = s.cur_scale;
        r.overflow = s.last_skipped;
        r.scale_is_int = (uint32_t)s.scale_is_int;
        log[(s.cur_iter - 1) % log_capacity] = r;
    }
    st->cur_scale = s.cur_scale;
    st->cur_iter = s.cur_iter;
    st->last_overflow_iter = s.last_overflow_iter;
    st->adam_step = s.adam_step;
    st->skipped_steps = s.skipped_steps;
    st->cur_hysteresis = s.cur_hysteresis;
    st->scale_is_int = s.scale_is_int;
    st->overflow = s.overflow;
    st->last_skipped = s.last_skipped;
    st->beta1_t_next = s.beta1_t_next;
    st->beta2_t_next = s.beta2_t_next;
    st->bias_correction1_next = s.bias_correction1_next;
    st->bias_correction2_next = s.bias_correction2_next;
    st->operator_step = s.operator_step;
    st->beta1_t_cur = s.beta1_t_cur;
    st->beta2_t_cur = s.beta2_t_cur;
    st->beta1_t_rest = s.beta1_t_rest;
    st->beta2_t_rest = s.beta2_t_rest;
    st->operator_beta1 = s.operator_beta1;
    st->operator_beta2 = s.operator_beta2;
    st->pending_operator_step = s.pending_operator_step;
}

__global__ void __launch_bounds__(64)
    scaler_update_kernel(ps_step_state* st, int flag_mode, ps_scale_record* log, int64_t log_capacity, int64_t operator_calls)
{
    const ps_step_state before = *st;
    const bool overflow = flag_mode == PS_FLAG_FROM_DEVICE ? (before.overflow != 0) : (flag_mode != 0);
    const ps_step_state after = scaler_updated(before, overflow, operator_calls);
    if (threadIdx.x == 0) scaler_store(st, after, log, log_capacity);
}

// ------------------------------------------- a whole device-decided step in two launches
//
// Probe, update and scale update.  As three kernels the last one cannot begin before the update has ended, because the update's
// waves read the state that it replaces, and it is a chain of its own: load, powers of the betas, store, 3.5 us behind its launch.
// Here the probe's first workgroup copies what the update needs of the state into the caller's scratch memory, the update's waves
// read the copy, and the update's first workgroup replaces the state while the others work.
//
// Bound by two launches and their ramps up to some 512 Ki elements, then by memory.  A step through FP16Adam.step(), three launches /
// two: among others 128 Ki elements 8.7 / 7.0 us (the host's part), 512 Ki 9.0 / 6.8, 1 Mi 10.9 / 9.2, 4 Mi 25.6 / 21.5, 16 Mi 75.7 / 71.9,
// 64 Mi 306.9 / 304, 200 Mi 921.9 / 922.3; waited for 128 Ki 20.6 / 18.8, 1 Mi 24.5 / 21.7.
//
// What the probe finds goes to a word of the scratch that the step before has cleared: one of two, in turn (a workgroup of the update
// clears the word of the step to come while others still read this step's).  The state's own flag, which copies of gradients
// may have raised before, travels with the copy.

// The state as the probe found it, as far as the update needs it.  The operator's arithmetic takes the first 64 bytes, one line
// and one load: as a copy of the whole state, five lines of which every wave looked at, the update of 8 x 64 Mi
// elements took 2358 us instead of 2276.
struct OpenedStep {
    double cur_scale;
    float beta1, beta2, b1t_next, b2t_next, b1t_rest, b2t_rest;
    uint32_t overflow;
    uint32_t turn;    // steps & 1 of this step
    uint32_t hit[2];  // the probe of step number `steps` found an inf or a nan: [steps & 1]
    uint32_t pad[4];
    double beta1_f64, beta2_f64, bc1_next, bc2_next;
    uint32_t pad2[8];
};
static_assert(sizeof(OpenedStep) == 128, "two lines");

// What the workgroups of a step share (PS_STEP_SCRATCH_BYTES, the caller's, zero at first).
struct StepScratch {
    // steps in one launch: adam_small_step_kernel
    uint64_t epoch;  // launches so far
    uint64_t pad0[15];
    uint32_t tickets;  // 0 between launches
    uint32_t pad1[15];
    uint64_t dirty, clean;  // epoch + 1 of the latest launch that was marked so
    uint64_t pad2[6];
    // steps in two launches
    OpenedStep opened;
    uint64_t steps;  // so far
    uint64_t pad3[7];
};
static_assert(sizeof(StepScratch) == PS_STEP_SCRATCH_BYTES, "the caller's allocation");

// Workgroups in front of every chunk's tiles: the first of all opens or closes the step, the others leave at once.  Lists that stream past
// the caches: as many as there are shader engines (8 XCDs of 4), which workgroups go round, so that every tile runs where it runs
// without them; one / 32 200 Mi elements 924.3 / 922.3 us (921.9 without any, in three launches), 4 Mi 21.5 / 22.3.
template <bool NT>
constexpr uint32_t kInFront = NT ? 32 : 1;
__device__ __forceinline__ bool first_of_all() { return (blockIdx.x | blockIdx.y) == 0; }

// The probe's first workgroup.
__device__ __forceinline__ void open_step(const ps_step_state* st, StepScratch* x)
{
    const StateView sv = view_state(st);
    const uint32_t turn = (uint32_t)x->steps & 1u;
    if (threadIdx.x != 0) return;
    OpenedStep& o = x->opened;  // (hit is written by the others)
    o.cur_scale = sv.cur_scale;
    o.beta1 = sv.beta1, o.beta2 = sv.beta2;
    o.b1t_next = sv.b1t_next, o.b2t_next = sv.b2t_next;
    o.b1t_rest = sv.b1t_rest, o.b2t_rest = sv.b2t_rest;
    o.overflow = sv.overflow;
    o.turn = turn;
    o.beta1_f64 = sv.beta1_f64, o.beta2_f64 = sv.beta2_f64;
    o.bc1_next = sv.bc1_next, o.bc2_next = sv.bc2_next;
}
__device__ __forceinline__ void probe_commit(uint32_t hit, StepScratch* x)
{
    if (__builtin_expect(__any(hit != 0), 0) && threadIdx.x == 0) x->opened.hit[x->steps & 1u] = 1u;
}

template <bool NT>
__global__ void __launch_bounds__(kScanBlock)
    open_even_chunks_kernel(const uint16_t* h16, uint32_t stride, uint32_t numel, uint32_t last, uint32_t short_by, const ps_step_state* st, StepScratch* x,
                            uint32_t keep)
{
    static_assert(kScanBlock == 64, "one wave");
    if (__builtin_expect(blockIdx.x < kInFront<NT>, 0)) {
        if (first_of_all()) open_step(st, x);
        return;
    }
    const uint32_t n = numel - (blockIdx.y == last ? short_by : 0u);
    probe_commit(probe_tile<NT>(h16 + (size_t)stride * blockIdx.y, n, blockIdx.x - kInFront<NT>, gridDim.x - kInFront<NT>, keep), x);
}

__global__ void __launch_bounds__(kScanBlock)
    open_chunks_kernel(ChunkBatch b, const ps_step_state* st, StepScratch* x)
{
    if (__builtin_expect(blockIdx.x < kInFront<false>, 0)) {
        if (first_of_all()) open_step(st, x);
        return;
    }
    probe_commit(scan_tile<uint16_t, kScanBlock, kScanUnroll>(b.c[blockIdx.y].param_fp16, b.n[blockIdx.y], blockIdx.x - kInFront<false>), x);
}

// What a wave of the update reads: the copy, with the flag as the probe left it.
template <int ARITH>
__device__ __forceinline__ StateView view_opened(const OpenedStep* __restrict__ x)
{
    StateView sv;
    sv.cur_scale = x->cur_scale;
    sv.beta1 = x->beta1, sv.beta2 = x->beta2;
    sv.b1t_next = x->b1t_next, sv.b2t_next = x->b2t_next;
    sv.b1t_rest = x->b1t_rest, sv.b2t_rest = x->b2t_rest;
    sv.overflow = x->overflow;
    uint32_t turn = x->turn, even = x->hit[0], odd = x->hit[1];
    if (ARITH == PS_ARITH_TORCH) {
        sv.beta1_f64 = x->beta1_f64, sv.beta2_f64 = x->beta2_f64;
        sv.bc1_next = x->bc1_next, sv.bc2_next = x->bc2_next;
    }
    ask_for(sv);
    asm volatile("" : "+s"(turn), "+s"(even), "+s"(odd));
    sv.overflow |= turn ? odd : even;
    return sv;
}

// The update's first workgroup.
struct Closing {
    ps_step_state* st;
    StepScratch* x;
    ps_scale_record* log;
    int64_t log_capacity, operator_calls;
};
__device__ __forceinline__ void close_step(const Closing& c)
{
    const ps_step_state now = *c.st;
    const uint64_t steps = c.x->steps;
    const uint32_t even = c.x->opened.hit[0], odd = c.x->opened.hit[1];
    const bool overflow = (now.overflow | (steps & 1u ? odd : even)) != 0;
    const ps_step_state after = scaler_updated(now, overflow, c.operator_calls);
    if (threadIdx.x == 0) {
        scaler_store(c.st, after, c.log, c.log_capacity);
        c.x->opened.hit[~steps & 1u] = 0;
        c.x->steps = steps + 1;
    }
}

template <int ARITH, int WD, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_even_chunks_closing_kernel(float* p32, float* m32, float* v32, uint16_t* h16, uint32_t stride, uint32_t numel, uint32_t last,
                                    uint32_t short_by, const OpenedStep* __restrict__ x, size_t chunk_numel, GatedArgs ga, FirstCall fc, Closing c)
{
    if (__builtin_expect(blockIdx.x < kInFront<NT>, 0)) {
        if (first_of_all()) close_step(c);
        return;
    }
    const EvenChunk t = even_chunk(p32, m32, v32, h16, stride, numel, last, short_by);
    const StateView sv = view_opened<ARITH>(x);
    even_gated_tile<ARITH, WD, NT>(t, blockIdx.x - kInFront<NT>, chunk_numel, ga, fc, sv);
}

template <int ARITH, int WD>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_chunks_closing_kernel(const OpenedStep* __restrict__ x, ChunkBatch b, size_t chunk_numel, GatedArgs ga, FirstCall fc, Closing c)
{
    if (__builtin_expect(blockIdx.x < kInFront<false>, 0)) {
        if (first_of_all()) close_step(c);
        return;
    }
    const uint32_t tile = blockIdx.x - kInFront<false>;
    const TileSource t = tile_source(b.c[blockIdx.y], b.n[blockIdx.y]);
    const CallSpan s = call_span(fc, tile);
    const StateView sv = view_opened<ARITH>(x);
    gated_tile<ARITH, WD, false>(t, tile, s, chunk_numel, ga, fc, sv);
}

// The same for a step whose tensors carry their own numbers, over tensors at the same place of their four lists: the probe's first
// workgroup forms the constants as well (plan_consts), which are ready long before the probe of the lists that this is for has ended;
// every launch of the update reads the copy, the first one closes the step.
//
// Device time of a step in a graph, four launches (probe, constants, update, scale update) / two, modules of BERT blocks with a rate per layer:
// 268 K elements 11.9 / 8.5 us, 2.1 M 17.6 / 16.4, 5.3 M 33.1 / 30.1, 43 M 205 / 197, 109 M 498 / 491, 223 M 1014 / 1009.  Bound by the launches and the
// chain of the constants up to some 1 M elements, then by memory.  Of the probe's lists only addresses and lengths travel, so that 48
// distinct calls fit beside them; steps with more, and tensors with binary32 gradients, take the launches one by one.
constexpr int kOpenClasses = 48;
struct ProbeList {
    const uint16_t* h[kBatch];
    uint32_t n[kBatch];
};

template <bool NT>
__global__ void __launch_bounds__(kScanBlock)
    open_planned_kernel(ProbeList b, PlanBatchOf<kOpenClasses> pb, PlanArgs a, ps_step_state* st, StepScratch* x, PlannedConsts* table, uint32_t keep)
{
    if (__builtin_expect(blockIdx.x < kInFront<NT>, 0)) {
        if (!first_of_all()) return;
        open_step(st, x);
        plan_consts(pb, a, st, table);
        return;
    }
    probe_commit(probe_tile<NT>(b.h[blockIdx.y], b.n[blockIdx.y], blockIdx.x - kInFront<NT>, gridDim.x - kInFront<NT>, keep), x);
}
static_assert(sizeof(ProbeList) + sizeof(PlanBatchOf<kOpenClasses>) + sizeof(PlanArgs) + 32 <= 4096, "kernel arguments of one launch");

template <int ARITH, int WD, bool NT>
__global__ void __launch_bounds__(kBlock) PS_OCCUPANCY
    adam_tensors_planned_closing_kernel(NearBatch b, const PlannedConsts* __restrict__ consts, const OpenedStep* __restrict__ x, Closing c)
{
    if (__builtin_expect(blockIdx.x < kInFront<NT>, 0)) {
        if (blockIdx.x == 0 && c.st != nullptr) close_step(c);  // (nullptr: a launch before this one has)
        return;
    }
    planned_tensor<ARITH, WD, NT>(tensor_view(b, blockIdx.x - kInFront<NT>), consts, [&]() {
        return (x->overflow | (x->turn ? x->hit[1] : x->hit[0])) != 0;
    });
}

// ------------------------------------------- a whole device-decided step over a short chunk list
//
// Probe, update (or restore) and scale update in one launch.  As three kernels they take three launches whatever the list's
// length, and the GPU waits for each.  The list is divided among workgroups of 15 waves with a tile (256 elements) each and a
// sixteenth that forms the step's constants and the next state.  EVERY workgroup probes the whole list, so that none has to
// wait for another.
//
// No workgroup waits, so the order in which they run is open, and one that starts late can find fp16 gradients already
// replaced by parameters.  What it finds then must not mislead it:
//   * clean step: a parameter that is inf or nan as binary16 looks like an overflow.  The wave that stores such a one first marks
//     the step as clean (StepScratch::clean); who finds an overflow looks there before it believes it.
//   * overflow: the gradient that says so may have been replaced.  A workgroup that has found it marks the step
//     (StepScratch::dirty) before it restores anything; who finds no overflow looks there before it believes it.
// A mark is stored with device scope and complete before the stores it announces are issued; a look is a device-scope load
// that depends on what the probe's loads brought.  Whoever has read a replaced value therefore sees the mark that came before it, and by
// induction over the workgroups' decisions all of them decide what the gradients alone say.  Marks carry the number
// of the launch (StepScratch::epoch), so nobody has to clear them.
//
// The state is replaced by the workgroup that took the last ticket; a ticket is taken when a workgroup has the state in its
// registers.  Tickets and looks cost a trip to memory each, in the shadow of the probe and of the arithmetic.  A list
// that one workgroup does alone needs neither, and no scratch.
//
// Bound by one CU's reads of the whole list (133 GB/s, 3.1 us for every 800 tiles) and by a chain of trips to memory: arguments,
// state or gradients, mark, stores.  A step through FP16Adam.step() among others, two launches / this: 73 tiles 6.9 / 5.8 us, 120
// 7.2 / 6.2, 180 7.2 / 6.5, 240 7.1 / 6.6, 300 7.2 / 6.9, 360 7.2 / 7.0; waited for 73 tiles 18.3 / 17.8, 180 18.7 / 18.6, 240 18.5 / 18.5, 300
// 18.3 / 18.7, 360 18.2 / 19.2.  The line (kSmallTiles) lies where neither is the longer one.  (By one workgroup 75 tiles took 12.45.)
// Device time in workgroups of 4 / 6 / 8 / 12 / 16 waves, with the state in memory (scaler_store): 75 tiles 7.6 / 6.9 / 6.6 / 7.2 / 6.9, 480
// tiles 15.2 / 12.1 / 10.9 / 9.5 / 9.5; two or four tiles a wave 480 tiles 9.8 / 13.8.
constexpr int kSmallWaves = PS_SMALL_WAVES;
constexpr uint32_t kSmallSpan = kSmallWaves - 1;  // tiles that a workgroup has in hand at a time
constexpr uint32_t kSmallScan = 4096;             // halves that a wave probes at a time: eight 16-byte loads a lane
constexpr unsigned kSmallTiles = PS_SMALL_TILES, kSmallTilesAlone = PS_SMALL_TILES_ALONE;
struct SmallStep {
    uint32_t tiles, n_tiles;  // of one chunk (as wide as the widest, like the grid of the chunk-list kernels), of the list
    uint32_t per_tile;        // 2^32 / tiles, rounded up: t * per_tile / 2^32 is t / tiles for every t of so short a list; 0: one tile each
    uint32_t scans, n_scans, per_scan;  // the same in spans of kSmallScan; n_scans 0: no probe
    size_t chunk_numel;
    ps_scale_record* log;
    int64_t log_capacity, operator_calls;
};

// The chunks of an EvenChunk list: 48 bytes of arguments where ChunkBatch has 2560, which cost the host 0.35 us a launch (the smoke
// test's list, 13.8 -> 13.4 us a step among others) and the kernel 0.4.
struct EvenBatch {
    ps_chunk first;
    uint32_t stride, numel, last, short_by;
};
__device__ __forceinline__ void small_chunk(const ChunkBatch& b, uint32_t k, ps_chunk& c, uint32_t& numel)
{
    c = b.c[k];
    numel = (uint32_t)b.n[k];
}
__device__ __forceinline__ void small_chunk(const EvenBatch& b, uint32_t k, ps_chunk& c, uint32_t& numel)
{
    const size_t at = (size_t)b.stride * k;
    c = ps_chunk{b.first.param_fp32 + at, b.first.exp_avg + at, b.first.exp_avg_sq + at, b.first.param_fp16 + at};
    numel = b.numel - (k == b.last ? b.short_by : 0u);
}

// ---- the probe: a binary16 value times zero is a NaN iff it is inf or nan, and a NaN stays one through every sum: one packed
// instruction for two values, where the masks of nonfinite_halves take seven.  (The probe of a list that is read once by the
// whole GPU hides them; here a CU reads all of it.)
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
struct SmallScan {
    uint4v w[kSmallScan / 512];
    uint32_t odd;
};
template <typename LIST>
__device__ __forceinline__ void small_scan_load(SmallScan& r, const LIST& b, const SmallStep& a, uint32_t i)
{
    // each workgroup begins somewhere else: all of them at the same lines of one L2 channel take their time
    uint32_t s = i + blockIdx.x;
    while (s >= a.n_scans) s -= a.n_scans;
    const uint32_t k = a.per_scan ? __umulhi(s, a.per_scan) : s, base = (s - k * a.scans) * kSmallScan;
    ps_chunk chunk;
    uint32_t numel;
    small_chunk(b, k, chunk, numel);
    r.odd = 0;
#pragma unroll
    for (uint32_t u = 0; u < kSmallScan / 512; ++u) r.w[u] = uint4v{0, 0, 0, 0};
    if (base >= numel) return;
    const PS_GLOBAL char* h = (const PS_GLOBAL char*)(chunk.param_fp16 + base);
    const uint32_t here = numel - base < kSmallScan ? numel - base : kSmallScan, n_vec = here / 8, behind = 8 * n_vec + threadIdx.x;
    // lanes behind the end read what is in front of it again
    if (n_vec != 0) {
#pragma unroll
        for (uint32_t u = 0; u < kSmallScan / 512; ++u) {
            const uint32_t v = u * 64 + threadIdx.x;
            r.w[u] = *(const PS_GLOBAL uint4v_half_aligned*)(h + (v < n_vec ? v : n_vec - 1) * 16);
        }
    }
    r.odd = *(const PS_GLOBAL uint16_t*)(h + (behind < here ? behind : here - 1) * 2);
}
__device__ __forceinline__ half2v small_scan_add(const SmallScan& r, half2v sum)
{
    const half2v zero = {0, 0};
#pragma unroll
    for (uint32_t u = 0; u < kSmallScan / 512; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t two = r.w[u][k];  // (a bit_cast of the vector's element is one of its first)
            sum = __builtin_elementwise_fma(__builtin_bit_cast(half2v, two), zero, sum);
        }
    return __builtin_elementwise_fma(__builtin_bit_cast(half2v, r.odd), zero, sum);
}

// ---- one lane's share of a tile: elements base + 4 * lane + e of a whole one, base + lane + 64 * e of any other
struct SmallShare {
    ps_chunk c;             // addresses of the tile's first element
    uint32_t base, numel;   // the tile's first element in its chunk; the chunk's elements
    uint32_t end;           // of what is updated, counted from base
    bool whole, here;       // with vector accesses; its chunk holds elements of the step's first operator call
    uint32_t g[4], h[4];    // g of a whole tile: two words of pairs, as they were loaded
    float old[4], p[4], m[4], v[4];
};
template <typename T>
__device__ __forceinline__ PS_GLOBAL T* small_at(const void* first, uint32_t i)
{
    return (PS_GLOBAL T*)((PS_GLOBAL char*)first + i * (uint32_t)sizeof(T));
}

// Elements of a tile that is not whole: all in flight; lanes behind the end read the last element again and store nothing.
__device__ __forceinline__ void small_load_single(SmallShare& o)
{
    if (o.end == 0) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t at = threadIdx.x + e * kBlock, i = at < o.end ? at : o.end - 1;
        o.g[e] = *small_at<uint16_t>(o.c.param_fp16, i);
        o.old[e] = *small_at<float>(o.c.param_fp32, i);
        o.m[e] = *small_at<float>(o.c.exp_avg, i);
        o.v[e] = *small_at<float>(o.c.exp_avg_sq, i);
    }
}

template <typename LIST>
__device__ __forceinline__ void small_load(SmallShare& o, const LIST& b, const SmallStep& a, const FirstCall& fc, uint32_t t)
{
    const uint32_t k = a.per_tile ? __umulhi(t, a.per_tile) : t, tile = t - k * a.tiles;
    small_chunk(b, k, o.c, o.numel);
    o.base = tile * kTile;
    o.c.param_fp32 += o.base;
    o.c.exp_avg += o.base;
    o.c.exp_avg_sq += o.base;
    o.c.param_fp16 += o.base;
    o.here = fc.chunk == (int)k;
    const bool cut = o.here && tile >= fc.lo_tile && tile < fc.hi_tile && !(tile >= fc.in_lo && tile < fc.in_hi);
    o.whole = o.base + kTile <= o.numel && !cut && aligned16(o.c.param_fp32, o.c.exp_avg, o.c.exp_avg_sq, o.c.param_fp16);
    if (o.whole) {
        o.end = kTile;
        const uint2v g = *small_at<uint2v>(o.c.param_fp16, threadIdx.x);
        const float4v p = *small_at<float4v>(o.c.param_fp32, threadIdx.x), m = *small_at<float4v>(o.c.exp_avg, threadIdx.x),
                      v = *small_at<float4v>(o.c.exp_avg_sq, threadIdx.x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o.g[e] = g[e & 1];
            o.old[e] = p[e], o.m[e] = m[e], o.v[e] = v[e];
        }
        return;
    }
    o.end = o.base >= o.numel ? 0 : o.numel - o.base < kTile ? o.numel - o.base : kTile;
    small_load_single(o);
}

template <int ARITH, int WD, int UNS>
__device__ __forceinline__ void small_math(SmallShare& o, const StepConsts& c, const FirstCall& fc)
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const size_t i = o.base + (o.whole ? 4 * threadIdx.x + e : threadIdx.x + e * kBlock);
        const bool first = o.here && i >= fc.lo && i < fc.hi;
        const float g = half_bits_to_float((o.whole ? o.g[e >> 1] >> (16 * (e & 1)) : o.g[e]) & 0xFFFFu);
        o.p[e] = o.old[e];
        adam_element<ARITH, WD, UNS>(c, first ? c.first_step_size : c.step_size, first ? c.first_bc2inv : c.bc2inv, g, o.p[e], o.m[e], o.v[e]);
        o.h[e] = float_to_half_bits(o.p[e]);
    }
}

// The constants of the step as the workgroup's waves share them.
struct SmallConsts {
    StepConsts c;
    int keeps_zeros_here, keeps_zeros;  // zeros_are_a_fixed_point, of chunks with and without elements of the first call
};
template <int ARITH, int WD>
__device__ __forceinline__ void small_update(SmallShare& o, const SmallConsts& k, const SmallStep& a, const FirstCall& fc)
{
    if (!o.whole && o.base + kTile > o.numel && o.numel < a.chunk_numel && !(o.here ? k.keeps_zeros_here : k.keeps_zeros)) {
        // the padding is computed, as in gated_tile
        o.end = (uint32_t)(a.chunk_numel - o.base < kTile ? a.chunk_numel - o.base : kTile);
        small_load_single(o);
    }
    if (k.c.unscale == UNSCALE_MUL)
        small_math<ARITH, WD, UNSCALE_MUL>(o, k.c, fc);
    else if (ARITH == PS_ARITH_OPERATOR && k.c.unscale == UNSCALE_DIV)
        small_math<ARITH, WD, UNSCALE_DIV>(o, k.c, fc);
    else
        small_math<ARITH, WD, UNSCALE_NONE>(o, k.c, fc);
}

__device__ __forceinline__ void small_store(const SmallShare& o)
{
    if (o.whole) {
        *small_at<float4v>(o.c.param_fp32, threadIdx.x) = float4v{o.p[0], o.p[1], o.p[2], o.p[3]};
        *small_at<float4v>(o.c.exp_avg, threadIdx.x) = float4v{o.m[0], o.m[1], o.m[2], o.m[3]};
        *small_at<float4v>(o.c.exp_avg_sq, threadIdx.x) = float4v{o.v[0], o.v[1], o.v[2], o.v[3]};
        *small_at<uint2v>(o.c.param_fp16, threadIdx.x) = uint2v{o.h[0] | (o.h[1] << 16), o.h[2] | (o.h[3] << 16)};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t i = threadIdx.x + e * kBlock;
        if (i >= o.end) continue;
        *small_at<float>(o.c.param_fp32, i) = o.p[e];
        *small_at<float>(o.c.exp_avg, i) = o.m[e];
        *small_at<float>(o.c.exp_avg_sq, i) = o.v[e];
        *small_at<uint16_t>(o.c.param_fp16, i) = (uint16_t)o.h[e];
    }
}

// fp16 <- RNE(fp32): a skipped step.  (`end` is still that of the chunk's elements.)
__device__ __forceinline__ void small_restore(const SmallShare& o)
{
    uint32_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = float_to_half_bits(o.old[e]);
    if (o.whole) {
        *small_at<uint2v>(o.c.param_fp16, threadIdx.x) = uint2v{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t i = threadIdx.x + e * kBlock;
        if (i < o.end && o.base + i < o.numel) *small_at<uint16_t>(o.c.param_fp16, i) = (uint16_t)h[e];
    }
}

// Stores with device scope, complete before anything behind it is issued.
__device__ __forceinline__ void small_mark(uint64_t* mark, uint64_t epoch)
{
    if (threadIdx.x == 0) __hip_atomic_store(mark, epoch + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");
}

// __syncthreads() for what crosses the waves here, LDS words: loads, stores and the ticket in flight are not waited for.
__device__ __forceinline__ void small_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    asm volatile("" ::: "memory");  // nor does the compiler move a load or store across
}

template <typename LIST, int ARITH, int WD>
__global__ void __launch_bounds__(64 * kSmallWaves)
    adam_small_step_kernel(LIST b, SmallStep a, GatedArgs ga, FirstCall fc, ps_step_state* st, StepScratch* scratch)
{
    static_assert(kBlock == 64 && kTile == 256, "tiles of one wave, four elements per lane");
    __shared__ uint32_t wave_hit[64];
    __shared__ uint32_t flagged, verdict, mark_low, mark_high;
    __shared__ SmallConsts consts;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.y), lane = threadIdx.x;
    const bool several = gridDim.x > 1;
    if (wave == kSmallSpan) {
        // ---- the state's wave
        const ps_step_state now = *st;
        uint64_t epoch = 0;
        uint32_t ticket = 0;
        const StateView sv = view_state(&now);
        if (several) {
            epoch = scratch->epoch;
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // all of the state is here: behind the ticket it may change
            PS_GLOBAL uint32_t* tickets = (PS_GLOBAL uint32_t*)&scratch->tickets;
            asm volatile("" : "+v"(tickets));  // (of an address known to be uniform the compiler waits for the result at once)
            if (lane == 0) ticket = __hip_atomic_fetch_add(tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const StepConsts c_rest = gated_consts<ARITH>(ga, sv, false);
        StepConsts c = c_rest;
        // the first call's pair is formed if the list holds any of that call
        if (fc.chunk >= 0 && ARITH == PS_ARITH_OPERATOR && ga.n_calls > 1)
            bias_scalars((float)ga.lr, sv.b1t_next, sv.b2t_next, ga.bias_correction != 0, &c.first_step_size, &c.first_bc2inv);
        if (lane == 0) {
            consts.c = c;
            consts.keeps_zeros = zeros_are_a_fixed_point(c_rest);
            consts.keeps_zeros_here = zeros_are_a_fixed_point(c);
            flagged = sv.overflow;
            mark_low = (uint32_t)epoch, mark_high = (uint32_t)(epoch >> 32);
        }
        small_barrier();
        bool overflow = sv.overflow != 0 || __any(lane < kSmallSpan && wave_hit[lane] != 0);
        uint64_t mark = 0;
        const bool marks = several && a.n_scans != 0 && !sv.overflow;
        if (marks) mark = __hip_atomic_load(overflow ? &scratch->clean : &scratch->dirty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const ps_step_state clean = scaler_updated(now, false, a.operator_calls);  // while the mark is on its way
        if (marks) {
            const bool marked = mark == epoch + 1;
            if (overflow && !marked) small_mark(&scratch->dirty, epoch);
            overflow = overflow != marked;
        }
        if (lane == 0) verdict = overflow;
        small_barrier();
        if (several && (uint32_t)__builtin_amdgcn_readfirstlane(ticket) != gridDim.x - 1) return;
        const ps_step_state after = overflow ? scaler_updated(now, true, a.operator_calls) : clean;
        if (lane == 0) {
            scaler_store(st, after, a.log, a.log_capacity);
            if (several) {
                scratch->epoch = epoch + 1;
                __hip_atomic_store(&scratch->tickets, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        return;
    }
    // ---- a wave with tiles
    SmallShare o;
    SmallScan scan;
    half2v sum = {0, 0};
    uint32_t t = blockIdx.x * kSmallSpan + wave;
    const bool any_tile = t < a.n_tiles;
    if (wave < a.n_scans) small_scan_load(scan, b, a, wave);
    if (any_tile) small_load(o, b, a, fc, t);
    if (wave < a.n_scans) sum = small_scan_add(scan, sum);
    for (uint32_t i = wave + kSmallSpan; i < a.n_scans; i += kSmallSpan) {
        small_scan_load(scan, b, a, i);
        sum = small_scan_add(scan, sum);
    }
    const bool hit = __any(nonfinite_halves(__builtin_bit_cast(uint32_t, sum)) != 0);
    if (lane == 0) wave_hit[wave] = hit;
    small_barrier();
    const bool known = __builtin_amdgcn_readfirstlane(flagged) != 0;
    if (any_tile && !known) small_update<ARITH, WD>(o, consts, a, fc);
    small_barrier();
    const bool overflow = __builtin_amdgcn_readfirstlane(verdict) != 0;
    if (!any_tile) return;
    for (;;) {
        if (overflow) {
            small_restore(o);
        } else {
            if (several && a.n_scans != 0) {
                uint32_t odd = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) odd |= nonfinite_halves(o.h[e]);
                if (__builtin_expect(__any(odd != 0), 0)) small_mark(&scratch->clean, ((uint64_t)mark_high << 32) | mark_low);
            }
            small_store(o);
        }
        t += gridDim.x * kSmallSpan;
        if (t >= a.n_tiles) return;
        small_load(o, b, a, fc, t);
        if (!overflow) small_update<ARITH, WD>(o, consts, a, fc);
    }
}

}  // namespace

#endif  // PS_KERNELS_H
