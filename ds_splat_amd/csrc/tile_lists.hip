// Per-tile depth-ordered Gaussian lists without a 64-bit sort of all K keys.
//
// The order the blend kernels need is (tile, depth bits, Gaussian index): the order a stable
// sort of the (tile << 32 | depth) keys produces, because keys are emitted by ascending Gaussian
// index and a Gaussian touches a tile at most once.  The same order falls out of
//   1. a stable sort of the N Gaussians by their 32 depth bits (N is ~10x smaller than K),
//   2. emitting (tile slot, Gaussian) pairs in that depth order,
//   3. a STABLE partition of the K pairs by tile slot alone (2 passes of <= 8 bits).
// Keys with a negative depth carry tile field -1 in the 64-bit scheme and sort first by their
// unsigned depth bits; here they take slot 0 and real tiles move up by one, and the unsigned
// depth order of step 1 keeps their relative order.  HBM traffic: 6 or 8 bytes per pair written
// once and moved twice, instead of 12 bytes moved five times.
#include "dsx_common.h"

#include <algorithm>
#include <mutex>

namespace dsx
{

// One helper stream per device (default priority, created on first use, kept until the process
// ends): work that does not depend on the depth sort runs there, beside the sort's
// latency-bound passes.  Returns nullptr when no stream can be made (the caller then stays on
// its own stream).
static hipStream_t helper_stream()
{
    constexpr int kMaxDevices = 64;
    static std::mutex mutex;
    static hipStream_t streams[kMaxDevices] = {};
    static bool tried[kMaxDevices] = {};
    int device = 0;
    if(hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices)
        return nullptr;
    std::lock_guard<std::mutex> lock(mutex);
    if(!tried[device])
    {
        tried[device] = true;
        hipStream_t s = nullptr;
        if(hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess)
            streams[device] = s;
        else
            (void)hipGetLastError();
    }
    return streams[device];
}

// Bin size of the tile lists: one list per tile below 2048 tiles (a 256 x 256 image has 16 bins of
// 4 x 4, and its 1024 blend wavefronts, four per tile there, would each filter a list sixteen times
// the tile's own); from 2048 tiles on, bins of 4 x 4 tiles (a Gaussian's rectangle then touches a few
// bins instead of a dozen tiles, and emission and partition shrink accordingly), or of 8 x 8 where
// that brings the lists, slot 0 included, down to the 256 that ONE partition pass handles
// (1920 x 1080: 135 lists instead of 510; a 3840 x 2160 image needs two passes either way).
// list_bin != 0 (dsx_camera::list_bin) asks for bins of that many tiles a side instead.
ListGrid list_grid(int image_width, int image_height, int list_bin)
{
    ListGrid g;
    g.ntx = tiles_x(image_width);
    g.nty = tiles_y(image_height);
    int side = list_bin ? list_bin : 1;
    if(!list_bin && g.ntx * g.nty >= 2048)
    {
        auto lists = [&](int64_t b) { return ((g.ntx + b - 1) / b) * ((g.nty + b - 1) / b); };
        side = (slot_bits((int)std::min<int64_t>(lists(4), 1 << 30)) > 8 && slot_bits((int)lists(8)) <= 8) ? 8 : 4;
        // (a bin's slot shares its 32-bit word with the 16-bit tile mask: at most 65534 bins; images beyond
        // that, hundreds of megapixels, get larger bins or, failing that, per-tile lists with 32-bit slots)
        if(lists(side) + 1 > 65535)
            side = lists(8) + 1 <= 65535 ? 8 : 1;
    }
    g.shift = side == 8 ? 3 : (side == 4 ? 2 : (side == 2 ? 1 : 0));
    g.nbx = (g.ntx + side - 1) / side;
    g.nby = (g.nty + side - 1) / side;
    return g;
}

__device__ __forceinline__ uint32_t wave_incl_scan32(uint32_t v, int)
{
    return wave_incl_scan_u32(v);
}

// number of set bits of a wavefront mask below this lane
__device__ __forceinline__ uint32_t bits_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// lanes of the wavefront that hold the same digit of up to kMaxBits bits; uniform flow only
template <int kMaxBits>
__device__ __forceinline__ uint64_t match_digit(uint32_t d, int bits)
{
    uint32_t lo = 0xffffffffu, hi = 0xffffffffu;
#pragma unroll
    for(int b = 0; b < kMaxBits; ++b)
    {
        if(b >= bits) // uniform: narrower digits need fewer rounds
            break;
        uint32_t x = (uint32_t)(((int32_t)(d << (31 - b))) >> 31); // all ones where bit b is set
        asm volatile("" : "+v"(x)); // the ballot tests x itself (one compare), not a second copy of the bit
        const uint64_t m = __ballot(x != 0);
        lo &= ~((uint32_t)m ^ x);
        hi &= ~((uint32_t)(m >> 32) ^ x);
    }
    return ((uint64_t)hi << 32) | lo;
}

// ---------------------------------------------------------------------------------------
// histograms of every digit in one read (run-length merged: neighbouring keys often share a digit)
// ---------------------------------------------------------------------------------------
#ifndef DSX_HIST_BLOCKS
#define DSX_HIST_BLOCKS 512 // few workgroups: each ends with one global atomic per bin, which serialise per address
#endif
// 1024 threads share one LDS histogram: the kernel is bound by latency (3 M keys are few), so
// it wants many wavefronts per CU, while every further workgroup adds a flush of up to 1024
// contended global atomics (256 threads: 0.029 ms, 1024 threads: 0.020 ms at 3 M keys)
constexpr int kHist32Threads = 1024;
// (keys of a thread: few, so that small inputs are spread over many workgroups; 100 K keys with eight 12 us, with two 6)
constexpr int kHist32Items = 2;
constexpr int kDepthHistItems = 8; // (four: 300 K and 500 K keys 0.5 us less, 1 M 1 us more, 3 M 1.6 more)

template <typename KeyT>
__global__ __launch_bounds__(kHist32Threads) void hist32_kernel(const KeyT* __restrict__ keys, int64_t count,
                                                                const Digits32 plan,
                                                                uint32_t* __restrict__ global_hist)
{
    __shared__ uint32_t hist[kMaxPasses32 * kBins32];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    for(int j = tid; j < plan.passes * kBins32; j += kHist32Threads)
        hist[j] = 0;
    __syncthreads();
    const int64_t chunk = (int64_t)kHist32Threads * kHist32Items;
    const int64_t chunks = (count + chunk - 1) / chunk;
    uint32_t ones = 0; // all-ones keys of this thread: counted here, added to their bins at the end
    for(int64_t c = blockIdx.x; c < chunks; c += gridDim.x)
    {
        uint32_t s[kHist32Items];
        bool valid[kHist32Items];
#pragma unroll
        for(int it = 0; it < kHist32Items; ++it)
        {
            const int64_t i = c * chunk + it * kHist32Threads + tid;
            valid[it] = i < count;
            s[it] = valid[it] ? (uint32_t)__builtin_nontemporal_load(keys + i) : 0u;
        }
#pragma unroll
        for(int it = 0; it < kHist32Items; ++it)
        {
            // lower digits: plain LDS atomics (values differ from lane to lane).  The most
            // significant digit takes few values (the exponent byte of depths, the high bits of
            // a tile slot): one add per distinct value of the wavefront, after a ballot, because
            // LDS atomics on one address serialise.
            // The all-ones depth keys of Gaussians that emit nothing, a third of a typical scene,
            // share one bin in every digit: each thread counts its own in a register and the
            // wavefront adds the sum to those bins once, at the end (0.026 -> 0.022 ms; a ballot
            // and one add per wavefront and item was slower than letting the atomics serialise).
            if(valid[it] && s[it] == 0xffffffffu)
            {
                ++ones;
                valid[it] = false;
            }
            for(int p = 0; p + 1 < plan.passes; ++p)
                if(valid[it])
                    atomicAdd(&hist[p * kBins32 + ((s[it] >> plan.shift[p]) & plan.mask[p])], 1u);
            {
                const int p = plan.passes - 1;
                const uint32_t d = (s[it] >> plan.shift[p]) & plan.mask[p];
                uint64_t todo = __ballot(valid[it]);
                for(int round = 0; round < 8 && todo; ++round)
                {
                    const int leader = __builtin_ctzll(todo);
                    const uint32_t dl = (uint32_t)__builtin_amdgcn_readlane((int)d, leader);
                    const uint64_t same = __ballot(valid[it] && d == dl) & todo;
                    if(lane == leader)
                        atomicAdd(&hist[p * kBins32 + dl], (uint32_t)__popcll(same));
                    todo &= ~same;
                }
                // more than eight distinct values in the wavefront: the digit is not a
                // concentrated one after all, the rest goes the plain way
                if((todo >> lane) & 1)
                    atomicAdd(&hist[p * kBins32 + d], 1u);
            }
        }
    }
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        ones += __shfl_xor(ones, o, DSX_WAVE);
    if(lane == 0 && ones)
        for(int p = 0; p < plan.passes; ++p)
            atomicAdd(&hist[p * kBins32 + plan.mask[p]], ones);
    __syncthreads();
    for(int j = tid; j < plan.passes * kBins32; j += kHist32Threads)
        if(hist[j])
            atomicAdd(&global_hist[j], hist[j]);
}

// ---------------------------------------------------------------------------------------
// one digit pass (chained scan over tiles, decoupled look-back) for (uint32 key, uint32 value)
// ---------------------------------------------------------------------------------------
constexpr uint32_t kFlagAggregate32 = 1u << 30;
constexpr uint32_t kFlagInclusive32 = 2u << 30;
constexpr uint32_t kFlagMask32 = 3u << 30;
constexpr uint32_t kValueMask32 = ~kFlagMask32;
#ifndef DSX_LOOK32
#define DSX_LOOK32 4
#endif
constexpr int kLookBatch32 = DSX_LOOK32;

static_assert(kSortThreads32 >= kDepthBins, "one thread per digit");
static_assert(kSortThreads32 * kSortItemsMax32 <= 65535, "u16 ranks");

// A tile rectangle as the projection packs it (16-bit fields) in 32 bits: 8 bits each for first
// column, first row, width and height, for images of at most 255 x 255 tiles.  The depth's sign
// takes the first column's place: column 255 does not exist, and what reads the sorted rectangles
// wants only the pair count of a Gaussian behind the camera (all its pairs go to slot 0), so its
// first column and row are not carried.
constexpr int kRect32MaxTiles = 255;
__device__ __forceinline__ uint32_t rect_to_32(uint2 r)
{
    const uint32_t size = ((r.y & 0xffu) << 16) | (((r.y >> 16) & 0xffu) << 24);
    return (r.y >> 31) ? (0xffu | size) : ((r.x & 0xffu) | (((r.x >> 16) & 0xffu) << 8) | size);
}
__device__ __forceinline__ uint2 rect_from_32(uint32_t v)
{
    const bool behind = (v & 0xffu) == 0xffu;
    const uint32_t size = ((v >> 16) & 0xffu) | ((v >> 24) << 16);
    return behind ? make_uint2(0u, size | 0x80000000u) : make_uint2((v & 0xffu) | (((v >> 8) & 0xffu) << 16), size);
}

// What a pass does about the Gaussians' tile rectangles, which the emission wants in depth order.
// Either the last pass gathers them (gather_dst[position] = gather_src[value]; a pair whose key is
// kNoPairsKey gets a zero record without the read): 1.9 M random 8-byte reads that pull 128-byte
// lines.  Or every pass carries the rectangle as a second 32-bit value (kCarry): the first pass
// reads the rectangles in index order, packs them (pack_src), the passes in between move them like
// the values (carry_in -> carry_out), and the last pass unpacks into unpack_dst.
struct RectJob
{
    const uint2* gather_src;
    uint2* gather_dst;
    uint32_t last_value; // of those that gather_src has a record for
    const uint2* pack_src;
    const uint32_t* carry_in;
    uint32_t* carry_out;
    uint2* unpack_dst;
};

// vals_in == nullptr: the values are the input positions (iota).  keys_out == nullptr: the
// keys are not needed after this pass.  KeyT: uint32_t, or uint16_t for tile slots that fit.
// kBits = 9: a pass of the depth sort over a known range.  The first pass (kFirst) turns the keys into their distances from
// `first`, of which a key without pairs has none: it becomes `behind`, stands behind the digits in its tile, and its value goes to
// its final place, behind the `emitting` others in the order of the input (how many lie in the tiles before is those tiles' keys
// less the sum of the digits' counts that the chained scan brings).  Later passes see the others only.
// polls: of a status that is not there, before a tile gives up (below zero: it does not look at all).  Its keys' places are then wrong, and so is what it leaves to later
// passes: no place is taken beyond the last one, and no value for a record's index beyond the last one.
struct KeyRange
{
    uint32_t first, behind, emitting;
};
template <typename KeyT, int kSort32Threads, int kSort32Items, bool kCarry, int kBits, bool kFirst>
__device__ __forceinline__ void onesweep32_pass(
    const KeyT* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, KeyT* __restrict__ keys_out,
    uint32_t* __restrict__ vals_out, int64_t count, int shift, uint32_t mask, const uint32_t* __restrict__ hist_counts,
    uint32_t* status, uint32_t* tile_counter, uint32_t* error_flag, int polls, const RectJob rects,
    const KeyRange range)
{
    const uint2* __restrict__ gather_src = rects.gather_src;
    uint2* __restrict__ gather_dst = rects.gather_dst;
    constexpr int kBins = 1 << kBits;
    // digits of a thread, side by side (two from eleven bits on; their statuses are one 64-bit word then, so both are there or neither)
    constexpr int kOwn = kBins > kSort32Threads ? kBins / kSort32Threads : 1;
    constexpr int kOwners = kBins / kOwn;
    static_assert(kOwn <= 2 && (kOwn == 1 || !kFirst), "a status word");
    constexpr int kSort32Tile = kSort32Threads * kSort32Items;
    constexpr int kSort32Waves = kSort32Threads / DSX_WAVE;
    __shared__ uint32_t s_keys[kSort32Tile]; // reused for the values in the second round
    __shared__ __attribute__((aligned(16))) uint16_t s_whist[kSort32Waves][kBins];
    __shared__ uint32_t s_digit_start[kBins];
    __shared__ uint32_t s_before[kFirst ? kBins / DSX_WAVE : 1]; // keys of the tiles before, by the digits' wavefronts
    __shared__ uint32_t s_none[kFirst ? kSort32Waves : 1];       // this tile's keys without pairs, by wavefront
    __shared__ uint32_t s_gbase[kBins];
    __shared__ __attribute__((aligned(16))) uint32_t s_wave_tot[kOwners / DSX_WAVE];
    __shared__ __attribute__((aligned(16))) uint32_t s_hist_tot[kOwners / DSX_WAVE];
    __shared__ uint32_t s_tile;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;

    if(tid == 0)
        s_tile = atomicAdd(tile_counter, 1u);
    for(int j = tid; j < kSort32Waves * kBins / 8; j += kSort32Threads)
        reinterpret_cast<uint4*>(&s_whist[0][0])[j] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    const int64_t tile = s_tile;
    const int64_t tile_base = tile * kSort32Tile;
    const int tile_n = (int)min((int64_t)kSort32Tile, count - tile_base);
    const int bits = 32 - __builtin_clz(mask); // mask = 2^bits - 1, bits >= 1
    auto digit_of = [shift, bits](uint32_t k) { return __builtin_amdgcn_ubfe(k, (uint32_t)shift, (uint32_t)bits); };

    // ---- load the keys (striped inside each wavefront: coalesced, order = (item, lane)) -----
    // Registers are what limits the blocks per compute unit here, so a thread keeps little per
    // item: the key while it is ranked and the rank as 16 bits; the value is fetched only once the key registers are
    // free.
    uint32_t key[kSort32Items];
    uint32_t pos2[(kSort32Items + 1) / 2]; // two 16-bit positions per register
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        const int local = wave * (kSort32Items * 64) + it * 64 + lane;
        // Places past the end of the input (last tile only) hold all-ones keys: they take the
        // highest digit and, being last in tile order, rank behind every real key, so the real
        // keys' positions are what they would be without them and no phase needs a validity test
        // except the stores (tile position < tile_n).
        // (first pass: they are keys without pairs, behind the others of that kind)
        key[it] = kFirst ? range.behind : 0xffffffffu;
        if(local < tile_n)
        {
            key[it] = (uint32_t)__builtin_nontemporal_load(keys_in + tile_base + local);
            if(kFirst)
                key[it] = min(key[it] - range.first, range.behind);
        }
    }

    // ---- wave-local stable rank ------------------------------------------------------------
    uint16_t* wh = s_whist[wave];
    uint32_t none = 0; // keys without pairs so far
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        const uint32_t d = digit_of(key[it]);
        uint64_t m = match_digit<kBits>(d, bits);
        uint64_t m_none = 0;
        if(kFirst)
        {
            m_none = __builtin_amdgcn_ballot_w64(key[it] == range.behind);
            m = __builtin_amdgcn_inverse_ballot_w64(m_none) ? m_none : m & ~m_none;
        }
        const uint32_t below = (uint32_t)bits_below(m);
        uint32_t old = wh[d];
        if(kFirst)
        {
            old = __builtin_amdgcn_inverse_ballot_w64(m_none) ? none : old;
            none += (uint32_t)__popcll(m_none);
        }
        __builtin_amdgcn_wave_barrier();
        if(below == 0 && (!kFirst || !__builtin_amdgcn_inverse_ballot_w64(m_none)))
            wh[d] = (uint16_t)(old + (uint32_t)__popcll(m));
        __builtin_amdgcn_wave_barrier();
        if(it & 1)
            pos2[it >> 1] |= (old + below) << 16;
        else
            pos2[it >> 1] = old + below;
        // pin the packed form here and make the key opaque: otherwise the compiler carries each
        // item's digit, histogram address and old count into the next phase in registers of their own
        asm volatile("" : "+v"(pos2[it >> 1]), "+v"(key[it]));
    }
    if(kFirst && lane == 0)
        s_none[wave] = none;
    __syncthreads();

    // ---- per-digit totals of the tile (thread d <-> digit d), wave offsets, digit starts ----
    const bool digit_thread = tid < kOwners; // thread d owns digit d (bins above the mask stay empty)
    const int digit0 = kOwn * tid;
    uint32_t total[kOwn] = {};
    uint32_t hist_excl[kOwn] = {};
    auto store_status = [&](const uint32_t (&counts)[kOwn], uint32_t flag) {
        uint32_t* const mine = status + tile * kBins + digit0;
        if constexpr(kOwn == 2)
            __hip_atomic_store(reinterpret_cast<unsigned long long*>(mine),
                               (unsigned long long)(counts[1] | flag) << 32 | (counts[0] | flag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
            __hip_atomic_store(mine, counts[0] | flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if(digit_thread)
    {
#pragma unroll
        for(int w = 0; w < kSort32Waves; ++w)
#pragma unroll
            for(int q = 0; q < kOwn; ++q)
            {
                const uint32_t c = s_whist[w][digit0 + q];
                s_whist[w][digit0 + q] = (uint16_t)total[q];
                total[q] += c;
            }
        store_status(total, tile == 0 ? kFlagInclusive32 : kFlagAggregate32);
        uint32_t sum = 0, hsum = 0, hcount[kOwn];
#pragma unroll
        for(int q = 0; q < kOwn; ++q)
        {
            // the digit's place in the whole output: exclusive scan of the pass's histogram (every
            // tile redoes this scan; that is cheaper than a kernel launch of its own)
            hcount[q] = hist_counts[digit0 + q];
            sum += total[q];
            hsum += hcount[q];
        }
        const uint32_t incl = wave_incl_scan32(sum, lane);
        if(lane == 63)
            s_wave_tot[wave] = incl;
        const uint32_t hincl = wave_incl_scan32(hsum, lane);
        if(lane == 63)
            s_hist_tot[wave] = hincl;
        uint32_t before = incl - sum, hbefore = hincl - hsum;
#pragma unroll
        for(int q = 0; q < kOwn; ++q)
        {
            s_gbase[digit0 + q] = before; // wave-local exclusive prefix, completed after the barrier
            before += total[q];
            hist_excl[q] = hbefore;
            hbefore += hcount[q];
        }
    }
    __syncthreads();
    if(digit_thread)
    {
        // totals of the digit wavefronts before this one
        const uint32_t prefix = sum_of_waves_before<kOwners / DSX_WAVE>(s_wave_tot, wave);
        const uint32_t hprefix = sum_of_waves_before<kOwners / DSX_WAVE>(s_hist_tot, wave);
#pragma unroll
        for(int q = 0; q < kOwn; ++q)
        {
            s_digit_start[digit0 + q] = prefix + s_gbase[digit0 + q];
            hist_excl[q] += hprefix;
        }
    }
    __syncthreads();

    // places of the tile from `emitters` on (there are none after the first pass) hold what does not emit
    int emitters = tile_n;
    uint32_t none_start = 0; // where this wavefront's begin
    if(kFirst)
    {
        uint32_t all = 0;
#pragma unroll
        for(int w = 0; w < kSort32Waves; ++w)
        {
            const uint32_t c = s_none[w];
            none_start += w < wave ? c : 0u;
            all += c;
        }
        emitters = kSort32Tile - __builtin_amdgcn_readfirstlane((int)all); // (the places past the end are counted among them)
        none_start = (uint32_t)emitters + __builtin_amdgcn_readfirstlane(none_start);
    }

    // ---- keys into LDS in tile-sorted order ----------------------------------------------
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        const uint32_t d = digit_of(key[it]);
        uint32_t start = s_digit_start[d] + s_whist[wave][d];
        if(kFirst)
            start = key[it] == range.behind ? none_start : start;
        const uint32_t p = ((pos2[it >> 1] >> (16 * (it & 1))) & 0xffffu) + start;
        s_keys[p] = key[it];
        pos2[it >> 1] = (it & 1) ? ((pos2[it >> 1] & 0xffffu) | (p << 16)) : ((pos2[it >> 1] & 0xffff0000u) | p);
    }

    // ---- the values: in flight while the chained scan runs ---------------------------------
    uint32_t val[kSort32Items];
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        const int local = wave * (kSort32Items * 64) + it * 64 + lane;
        val[it] = 0;
        if(local < tile_n)
            val[it] = vals_in ? __builtin_nontemporal_load(vals_in + tile_base + local) : (uint32_t)(tile_base + local);
    }
    uint32_t carried[kCarry ? kSort32Items : 1];
    if(kCarry)
    {
#pragma unroll
        for(int it = 0; it < kSort32Items; ++it)
        {
            const int local = wave * (kSort32Items * 64) + it * 64 + lane;
            carried[it] = 0;
            if(local < tile_n)
                carried[it] = rects.pack_src ? rect_to_32(rects.pack_src[tile_base + local])
                                             : __builtin_nontemporal_load(rects.carry_in + tile_base + local);
        }
    }

    // ---- chained scan over earlier tiles (decoupled look-back), one thread per digit -------
    if(digit_thread)
    {
        uint32_t excl[kOwn] = {};
        if(tile > 0 && (uint32_t)digit0 <= mask) // bins above the mask are empty in every tile
        {
            int64_t t = tile - 1; // next predecessor to account for
            int spins = 0;
            bool done = polls < 0;
            if(done)
                *error_flag = 1u;
            while(!done)
            {
                uint32_t v[kLookBatch32][kOwn];
#pragma unroll
                for(int b = 0; b < kLookBatch32; ++b)
                {
                    // rows below tile 0 are read as tile 0, whose status is inclusive from the start
                    const int64_t row = t - b > 0 ? t - b : 0;
                    uint32_t* const theirs = status + row * kBins + digit0;
                    if constexpr(kOwn == 2)
                    {
                        const unsigned long long both =
                            __hip_atomic_load(reinterpret_cast<unsigned long long*>(theirs), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        v[b][0] = (uint32_t)both;
                        v[b][kOwn - 1] = (uint32_t)(both >> 32);
                    }
                    else
                        v[b][0] = __hip_atomic_load(theirs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for(int b = 0; b < kLookBatch32; ++b)
                {
                    if(done)
                        break;
                    if((v[b][0] & kFlagMask32) == 0)
                    {
                        if(++spins > polls)
                        {
                            *error_flag = 1u;
                            done = true;
                        }
                        else
                            __builtin_amdgcn_s_sleep(1);
                        break;
                    }
#pragma unroll
                    for(int q = 0; q < kOwn; ++q)
                        excl[q] += v[b][q] & kValueMask32;
                    --t;
                    if(v[b][0] & kFlagInclusive32)
                        done = true;
                }
            }
            uint32_t all[kOwn];
#pragma unroll
            for(int q = 0; q < kOwn; ++q)
                all[q] = (excl[q] + total[q]) & kValueMask32;
            store_status(all, kFlagInclusive32);
        }
#pragma unroll
        for(int q = 0; q < kOwn; ++q)
            s_gbase[digit0 + q] = hist_excl[q] + excl[q] - s_digit_start[digit0 + q];
        if(kFirst)
        {
            const uint32_t before = wave_sum_u32(excl[0]);
            if(lane == 0)
                s_before[wave] = before;
        }
    }
    __syncthreads();
    uint32_t tail = 0; // place of the tile's first key without pairs, less its position in the tile
    if(kFirst)
    {
        tail = range.emitting + (uint32_t)tile_base - (uint32_t)emitters;
#pragma unroll
        for(int w = 0; w < kBins / DSX_WAVE; ++w)
            tail -= s_before[w];
        tail = __builtin_amdgcn_readfirstlane(tail);
    }

    // ---- scatter keys: consecutive threads -> consecutive addresses inside a digit's run ----
    const uint32_t last_place = (uint32_t)(count - 1);
    uint32_t out[kSort32Items];            // where the key at tile position it * threads + tid goes
    uint32_t no_record = 0;                // bit it: that key is kNoPairsKey (its record is known to be zero)
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        const int j = it * kSort32Threads + tid;
        if((it & 3) == 0)
            __builtin_amdgcn_sched_barrier(0); // four items in flight at a time: registers, not latency, are scarce
        if(j < tile_n)
        {
            const uint32_t kk = s_keys[j];
            const uint32_t digit_base = s_gbase[digit_of(kk)];
            out[it] = min((!kFirst || j < emitters ? digit_base : tail) + (uint32_t)j, last_place);
            if(gather_src && kk == kNoPairsKey)
                no_record |= 1u << it;
            if(keys_out && (!kFirst || j < emitters))
                keys_out[out[it]] = (KeyT)kk;
        }
    }
    __syncthreads();

    // ---- values through the same buffer, same positions ------------------------------------
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        s_keys[(pos2[it >> 1] >> (16 * (it & 1))) & 0xffffu] = val[it];
    }
    __syncthreads();
#pragma unroll
    for(int it = 0; it < kSort32Items; ++it)
    {
        const int j = it * kSort32Threads + tid;
        if((it & 3) == 0)
            __builtin_amdgcn_sched_barrier(0);
        if(j < tile_n)
        {
            const uint32_t v = s_keys[j];
            vals_out[out[it]] = v;
            // optional: a per-value record follows its value to the sorted position (the random
            // gather overlaps with the scatter traffic of the pass)
            if(gather_src)
                gather_dst[out[it]] = ((no_record >> it) & 1u) ? make_uint2(0u, 0u) : gather_src[min(v, rects.last_value)];
        }
    }
    if(kCarry)
    {
        // ---- the carried rectangles through the same buffer, same positions ------------------
        __syncthreads();
#pragma unroll
        for(int it = 0; it < kSort32Items; ++it)
            s_keys[(pos2[it >> 1] >> (16 * (it & 1))) & 0xffffu] = carried[it];
        __syncthreads();
#pragma unroll
        for(int it = 0; it < kSort32Items; ++it)
        {
            const int j = it * kSort32Threads + tid;
            if((it & 3) == 0)
                __builtin_amdgcn_sched_barrier(0);
            if(kFirst ? j < emitters : j < tile_n)
            {
                const uint32_t v = s_keys[j];
                if(rects.unpack_dst)
                    rects.unpack_dst[out[it]] = rect_from_32(v);
                else
                    rects.carry_out[out[it]] = v;
            }
        }
    }
}

// (eight wavefronts per SIMD: two workgroups per compute unit with digits of eight and nine bits, whatever the tile, and of ten with up to eight
// keys a thread; 88 KB of LDS with ten bits and twelve keys, and what eleven bits take, leave room for one)
template <typename KeyT, int kSort32Threads, int kSort32Items, bool kCarry, int kBits>
__global__ __launch_bounds__(kSort32Threads) __attribute__((amdgpu_waves_per_eu(8))) void onesweep32_kernel(
    const KeyT* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, KeyT* __restrict__ keys_out,
    uint32_t* __restrict__ vals_out, int64_t count, int shift, uint32_t mask, const uint32_t* __restrict__ hist_counts,
    uint32_t* status, uint32_t* tile_counter, uint32_t* error_flag, int polls, const RectJob rects)
{
    onesweep32_pass<KeyT, kSort32Threads, kSort32Items, kCarry, kBits, false>(
        keys_in, vals_in, keys_out, vals_out, count, shift, mask, hist_counts, status, tile_counter, error_flag, polls, rects,
        KeyRange{});
}

// the first pass of the depth sort over a known range
template <int kSort32Items, bool kCarry>
__global__ __launch_bounds__(kSortThreads32) __attribute__((amdgpu_waves_per_eu(8))) void onesweep32_first_kernel(
    const uint32_t* __restrict__ keys_in, uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out, int64_t count, int shift,
    uint32_t mask, const uint32_t* __restrict__ hist_counts, uint32_t* status, uint32_t* tile_counter, uint32_t* error_flag,
    int polls, const RectJob rects, const KeyRange range)
{
    onesweep32_pass<uint32_t, kSortThreads32, kSort32Items, kCarry, kDepthBits, true>(
        keys_in, nullptr, keys_out, vals_out, count, shift, mask, hist_counts, status, tile_counter, error_flag, polls, rects,
        range);
}

Sort32Workspace sort32_workspace(int64_t count, int key_bits, int tile_keys, bool wide)
{
    auto align = [](size_t x) { return (x + 255) & ~(size_t)255; };
    Sort32Workspace w;
    w.passes = wide ? 1 : digits32(key_bits).passes;
    w.tiles = (count + tile_keys - 1) / tile_keys;
    size_t off = 0;
    // (32 bits: perhaps a depth sort)
    const size_t words = wide ? (size_t)1 << key_bits : (key_bits == 32 ? kSortWordsMost : (size_t)w.passes * kBins32);
    w.hist = off;
    off = align(off + words * 4);
    w.counters = off;
    off = align(off + (size_t)(w.passes + 1) * 4);
    w.status = off;
    off = align(off + words * (size_t)w.tiles * 4);
    w.bytes = off;
    return w;
}

// zeroes histograms, tile counters and look-back statuses of one sort
// (extra_bytes: memory right behind the workspace that the same fill clears)
static int sort32_clear(int64_t count, int key_bits, int tile_keys, void* sort_ws, hipStream_t stream,
                        size_t extra_bytes = 0)
{
    const Sort32Workspace w = sort32_workspace(count, key_bits, tile_keys);
    return launch_fill_u32(reinterpret_cast<uint32_t*>(static_cast<char*>(sort_ws) + w.hist),
                           (int64_t)((w.bytes + extra_bytes) / 4), 0u, stream);
}

// The digit passes of a sort whose raw digit histograms are in `counts` (the workspace's own
// histogram area when counts is null).
// Ping-pong between (keys_a, vals_a) and (keys_b, vals_b); *keys_out / *vals_out say where the
// result is (keys only when keep_keys).
// gather_src / gather_dst: records that the last pass brings to the values' sorted positions by a
// gather.  carry_a / carry_b (with gather_src and gather_dst): the records travel through the passes
// as packed 32-bit values instead, in ping-pong buffers of their own (the first pass packs them from
// gather_src, the last one unpacks them into gather_dst).
template <typename KeyT, int kThreads, int kItems, bool kCarry = false, int kBits = kBits32>
static int sort32_passes(int64_t count, int key_bits, KeyT* keys_a, uint32_t* vals_a, KeyT* keys_b, uint32_t* vals_b,
                         bool iota_values, bool keep_keys, void* sort_ws, const char* label, hipStream_t stream,
                         KeyT** keys_out, uint32_t** vals_out, const uint2* gather_src = nullptr,
                         uint2* gather_dst = nullptr, const uint32_t* counts = nullptr, uint32_t* carry_a = nullptr,
                         uint32_t* carry_b = nullptr, int polls = kSpinLimit32)
{
    constexpr bool kWide = kBits > kBits32; // (one digit of kBits bits)
    const Sort32Workspace w = sort32_workspace(count, key_bits, kThreads * kItems, kWide);
    const Digits32 plan = kWide ? partition_digits(kBits, true) : digits32(key_bits);
    char* base = static_cast<char*>(sort_ws);
    uint32_t* hist = reinterpret_cast<uint32_t*>(base + w.hist);
    uint32_t* counters = reinterpret_cast<uint32_t*>(base + w.counters);
    uint32_t* status = reinterpret_cast<uint32_t*>(base + w.status);
    const uint32_t* raw = counts ? counts : (const uint32_t*)hist; // the passes scan their histogram themselves
    KeyT* kin = keys_a;
    uint32_t* vin = vals_a;
    KeyT* kout = keys_b;
    uint32_t* vout = vals_b;
    uint32_t* cin = carry_a;
    uint32_t* cout = carry_b;
    for(int p = 0; p < plan.passes; ++p)
    {
        const bool last = p == plan.passes - 1;
        RectJob job = {};
        if(kCarry)
        {
            job.pack_src = p == 0 ? gather_src : nullptr;
            job.carry_in = cin;
            job.carry_out = cout;
            job.unpack_dst = last ? gather_dst : nullptr;
        }
        else if(last)
        {
            job.gather_src = gather_src;
            job.gather_dst = gather_dst;
            job.last_value = (uint32_t)(count - 1);
        }
        {
            DSX_TIMED(label, stream);
            hipLaunchKernelGGL((onesweep32_kernel<KeyT, kThreads, kItems, kCarry, kBits>), dim3((unsigned)w.tiles), dim3(kThreads), 0,
                               stream, (const KeyT*)kin, (const uint32_t*)((p == 0 && iota_values) ? nullptr : vin),
                               (last && !keep_keys) ? (KeyT*)nullptr : kout, vout, count, plan.shift[p], plan.mask[p],
                               raw + p * kBins32, status + (size_t)p * w.tiles * kBins32,
                               counters + p, counters + w.passes, polls, job);
        }
        DSX_LAUNCH_CHECK();
        KeyT* tk = kin;
        kin = kout;
        kout = tk;
        uint32_t* tv = vin;
        vin = vout;
        vout = tv;
        uint32_t* tc = cin;
        cin = cout;
        cout = tc;
    }
    *keys_out = kin;
    *vals_out = vin;
    return DSX_OK;
}

// Stable ascending sort of `count` (key, value) pairs by the low key_bits bits of the key.
int launch_sort32(int64_t count, int key_bits, uint32_t* keys_a, uint32_t* vals_a, uint32_t* keys_b,
                  uint32_t* vals_b, bool iota_values, bool keep_keys, void* sort_ws, hipStream_t stream,
                  uint32_t** keys_out, uint32_t** vals_out, const uint2* gather_src, uint2* gather_dst,
                  bool already_cleared, uint32_t* carry_a, uint32_t* carry_b, int polls)
{
    *keys_out = keys_a;
    *vals_out = vals_a;
    if(count <= 0)
        return DSX_OK;
    if(count >= (1ll << 30))
        return DSX_ERR_TOO_LARGE;
    int rc = already_cleared ? DSX_OK : sort32_clear(count, key_bits, sort32_tile_keys(count), sort_ws, stream);
    if(rc)
        return rc;
    const Sort32Workspace w = sort32_workspace(count, key_bits, sort32_tile_keys(count));
    const int64_t chunks = (count + kHist32Threads * kHist32Items - 1) / (kHist32Threads * kHist32Items);
    {
        DSX_TIMED("hist32_kernel", stream);
        hipLaunchKernelGGL(hist32_kernel<uint32_t>, dim3((unsigned)min((int64_t)DSX_HIST_BLOCKS, chunks)), dim3(kHist32Threads), 0,
                           stream, (const uint32_t*)keys_a, count, digits32(key_bits),
                           reinterpret_cast<uint32_t*>(static_cast<char*>(sort_ws) + w.hist));
    }
    DSX_LAUNCH_CHECK();
    const bool carry = carry_a && carry_b && gather_src && gather_dst;
#define DSX_SORT32_ITEMS(ITEMS)                                                                                       \
    case ITEMS:                                                                                                       \
        return carry ? sort32_passes<uint32_t, kSortThreads32, ITEMS, true>(                                          \
                           count, key_bits, keys_a, vals_a, keys_b, vals_b, iota_values, keep_keys, sort_ws,          \
                           "onesweep32_kernel<sort>", stream, keys_out, vals_out, gather_src, gather_dst, nullptr,    \
                           carry_a, carry_b, polls)                                                                   \
                     : sort32_passes<uint32_t, kSortThreads32, ITEMS>(count, key_bits, keys_a, vals_a, keys_b, vals_b, \
                                                                      iota_values, keep_keys, sort_ws,                \
                                                                      "onesweep32_kernel<sort>", stream, keys_out,    \
                                                                      vals_out, gather_src, gather_dst, nullptr,      \
                                                                      nullptr, nullptr, polls)
    switch(sort32_items(count))
    {
        DSX_SORT32_ITEMS(1);
        DSX_SORT32_ITEMS(2);
        DSX_SORT32_ITEMS(3);
        DSX_SORT32_ITEMS(4);
        DSX_SORT32_ITEMS(6);
        DSX_SORT32_ITEMS(8);
        DSX_SORT32_ITEMS(kSortItemsMax32);
    }
#undef DSX_SORT32_ITEMS
    return DSX_ERR_RUNTIME;
}

// one of the words of pinned host memory that the host polls
__device__ __forceinline__ void store_to_host(const HostCounts& to, int word, unsigned long long count)
{
    constexpr unsigned long long most = 1ull << (kTicketShift - 1);
    __hip_atomic_store(to.words + word, (to.ticket << kTicketShift) | (count < most ? count : most), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// Sixteen bytes of an `order` buffer, whose address is a multiple of eight (that the rectangles and the 64-bit sums need too) and no more
struct __attribute__((packed, aligned(8))) Words4
{
    uint32_t x, y, z, w;
};
static_assert(sizeof(Words4) == 16, "one load");

// A thread's keys of one step through all of them, sixteen bytes at a time (the buffer is padded to whole lines)
constexpr int kBatchLoads = 4;
constexpr int kBatchKeys = 4 * kBatchLoads * kHist32Threads;
struct KeyBatch
{
    uint4 k[kBatchLoads];
};
__device__ __forceinline__ KeyBatch load_keys(const uint32_t* keys, int i0, int n)
{
    KeyBatch batch;
#pragma unroll
    for(int b = 0; b < kBatchLoads; ++b)
    {
        const int i = i0 + 4 * (b * kHist32Threads + (int)threadIdx.x);
        uint4 k = make_uint4(kNoPairsKey, kNoPairsKey, kNoPairsKey, kNoPairsKey);
        if(i < n)
        {
            const Words4 four = *reinterpret_cast<const Words4*>(keys + i);
            k = make_uint4(four.x, four.y, four.z, four.w);
        }
        if(i0 + kBatchKeys > n) // (uniform: the words behind the last key hold anything)
        {
            k.y = i + 1 < n ? k.y : kNoPairsKey;
            k.z = i + 2 < n ? k.z : kNoPairsKey;
            k.w = i + 3 < n ? k.w : kNoPairsKey;
        }
        batch.k[b] = k;
    }
    return batch;
}

// What a thread of `kThreads` finds in its share of the blocks' key ranges: the extremes, and how many keys emit.  Eight loads in
// flight: one after the other they are most of a short kernel's time.
struct KeySpan
{
    uint32_t near16 = 0, far16 = 0, emitting = 0;
};
template <int kThreads>
__device__ __forceinline__ KeySpan key_span(const uint2* __restrict__ ranges, int blocks)
{
    KeySpan s;
    for(int b0 = threadIdx.x; b0 < blocks; b0 += 8 * kThreads)
    {
        uint2 r[8];
#pragma unroll
        for(int u = 0; u < 8; ++u)
            r[u] = b0 + u * kThreads < blocks ? ranges[b0 + u * kThreads] : make_uint2(0u, 0u);
#pragma unroll
        for(int u = 0; u < 8; ++u)
        {
            s.near16 = max(s.near16, r[u].x & 0xffffu);
            s.far16 = max(s.far16, r[u].y);
            s.emitting += r[u].x >> 16;
        }
    }
    return s;
}

// Bins of equal width over a known range of depths, where that is narrow and more than a thin layer (which would crowd a few buckets);
// the bin of a distance from its first key
__host__ __device__ constexpr bool depth_bins(const DepthRange& range)
{
    return range.narrow && range.behind >= 16u << 16; // (an eighth of an octave)
}
__device__ __forceinline__ uint32_t depth_bin_scale(const DepthRange& range, int bin_bits)
{
    return (1u << (bin_bits + 16)) / (range.behind >> 16); // (2^bin_bits bins, 2^32 times, over the distances)
}
__device__ __forceinline__ uint32_t depth_bin(uint32_t distance, uint32_t scale)
{
    return __umulhi(distance, scale);
}

// The histograms of a depth sort whose range only the device knows yet: every workgroup finds it from the projection's
// blocks, the first one tells the host, and the digits are those of depth_range(); with bin_bits, where the range is narrow, one
// histogram of so many bins of the range, and what depth_scatter_kernel (launched only then) wants to know of the blocks, in `span`: the
// range's ends (the nearest one's complement), the emitting keys, a spare word, and how many of them lie in front of each of kSpanChunks
// chunks of blocks.
// (kBinsWorkgroups: that count bins; each adds them to memory, which takes some 45 additions a clock.  us at 3 M,
// beside the counting of the tiles: 366 43, 128 17, 64 22)
constexpr int kBinsWorkgroups = 128;
constexpr int kSpanWords = 4, kSpanChunks = kHist32Threads;
__host__ __device__ constexpr int span_chunk(int blocks) { return (blocks + kSpanChunks - 1) / kSpanChunks; }
__global__ __launch_bounds__(kHist32Threads) void depth_hist_kernel(const uint32_t* __restrict__ keys, int64_t count,
                                                                    const uint2* __restrict__ ranges, int64_t blocks,
                                                                    uint32_t* __restrict__ digit_hist,
                                                                    uint32_t* __restrict__ bin_hist, int bin_bits,
                                                                    uint32_t* __restrict__ span, const HostCounts to_host)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t hist[]; // of kSortWordsMost words, or the bins if they are more
    __shared__ uint2 s_range[kHist32Threads / DSX_WAVE];
    __shared__ uint32_t s_emitting[kHist32Threads / DSX_WAVE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for(int j = tid; j < max((int)kSortWordsMost, bin_bits ? 1 << bin_bits : 0); j += kHist32Threads)
        hist[j] = 0;
    const KeySpan mine = key_span<kHist32Threads>(ranges, (int)blocks);
    uint32_t near16 = wave_incl_max_scan(mine.near16), far16 = wave_incl_max_scan(mine.far16);
    const uint32_t emitting = wave_sum_u32(mine.emitting);
    if(lane == 63)
    {
        s_range[wave] = make_uint2(near16, far16);
        s_emitting[wave] = emitting;
    }
    __syncthreads();
#pragma unroll
    for(int w = 0; w < kHist32Threads / DSX_WAVE; ++w)
    {
        near16 = w == 0 ? s_range[0].x : max(near16, s_range[w].x);
        far16 = w == 0 ? s_range[0].y : max(far16, s_range[w].y);
    }
    const uint32_t lowest = 0xffffu - (uint32_t)__builtin_amdgcn_readfirstlane((int)near16);
    const uint32_t highest = (uint32_t)__builtin_amdgcn_readfirstlane((int)far16);
    if(blockIdx.x == 0 && tid == 0)
    {
        unsigned long long all = 0;
        for(int w = 0; w < kHist32Threads / DSX_WAVE; ++w)
            all += s_emitting[w];
        store_to_host(to_host, 2, lowest | ((unsigned long long)highest << 16));
        store_to_host(to_host, 3, all);
    }
    const DepthRange range = depth_range(lowest, highest);
    const int bins = range.narrow ? kDepthBins : kBins32;
    const bool by_bins = bin_bits != 0 && depth_bins(range);
    const uint32_t scale = by_bins ? depth_bin_scale(range, bin_bits) : 0u;
    if(blockIdx.x == 0 && by_bins)
    {
        const int chunk = span_chunk((int)blocks);
        uint32_t mine_emit = 0;
        for(int b = chunk * tid; b < min(chunk * (tid + 1), (int)blocks); ++b)
            mine_emit += ranges[b].x >> 16;
        const uint32_t incl = wave_incl_scan_u32(mine_emit);
        __syncthreads();
        if(lane == 63)
            s_emitting[wave] = incl;
        __syncthreads();
        uint32_t before = incl - mine_emit;
#pragma unroll
        for(int w = 0; w < kHist32Threads / DSX_WAVE; ++w)
            before += w < wave ? s_emitting[w] : 0u;
        span[kSpanWords + tid] = before;
        if(tid == kHist32Threads - 1)
        {
            span[0] = 0xffffu - lowest;
            span[1] = highest;
            span[2] = before + mine_emit;
        }
    }
    uint32_t none = 0; // keys without pairs: counted by their thread, added to their bins at the end (four digits; three leave them out)
    const int workgroups = by_bins ? min((int)gridDim.x, kBinsWorkgroups) : (int)gridDim.x;
    if((int)blockIdx.x >= workgroups)
        return;
    if(by_bins)
        for(int64_t i0 = (int64_t)blockIdx.x * kBatchKeys; i0 < count; i0 += (int64_t)workgroups * kBatchKeys)
        {
            const KeyBatch batch = load_keys(keys, (int)i0, (int)count);
#pragma unroll
            for(int b = 0; b < kBatchLoads; ++b)
            {
                const uint32_t four[4] = {batch.k[b].x, batch.k[b].y, batch.k[b].z, batch.k[b].w};
#pragma unroll
                for(int u = 0; u < 4; ++u)
                    if(four[u] != kNoPairsKey)
                        atomicAdd(&hist[depth_bin(four[u] - range.first, scale)], 1u);
            }
        }
    const int64_t chunk = (int64_t)kHist32Threads * kDepthHistItems, chunks = by_bins ? 0 : (count + chunk - 1) / chunk;
    for(int64_t c = blockIdx.x; c < chunks; c += gridDim.x)
    {
        uint32_t key[kDepthHistItems];
        bool valid[kDepthHistItems];
#pragma unroll
        for(int it = 0; it < kDepthHistItems; ++it)
        {
            const int64_t i = c * chunk + it * kHist32Threads + tid;
            valid[it] = i < count;
            key[it] = valid[it] ? __builtin_nontemporal_load(keys + i) : 0u;
        }
#pragma unroll
        for(int it = 0; it < kDepthHistItems; ++it)
        {
            if(valid[it] && key[it] == kNoPairsKey)
            {
                ++none;
                valid[it] = false;
            }
            // (the top digit takes few values only where the depths span many octaves: the keys go by distance here)
            if(valid[it])
#pragma unroll
                for(int p = 0; p < kMaxPasses32; ++p)
                    if(p < range.digits.passes)
                        atomicAdd(&hist[p * bins + (((key[it] - range.first) >> range.digits.shift[p]) & range.digits.mask[p])], 1u);
        }
    }
    none = range.narrow ? 0u : wave_sum_u32(none);
    if(lane == 0 && none)
#pragma unroll
        for(int p = 0; p < kMaxPasses32; ++p)
            if(p < range.digits.passes)
                atomicAdd(&hist[p * bins + ((range.behind >> range.digits.shift[p]) & range.digits.mask[p])], none);
    __syncthreads();
    uint32_t* const global_hist = by_bins ? bin_hist : digit_hist;
    for(int j = tid; j < (by_bins ? 1 << bin_bits : range.digits.passes * bins); j += kHist32Threads)
        if(hist[j])
            atomicAdd(&global_hist[j], hist[j]);
}

// ---------------------------------------------------------------------------------------
// depth order of the Gaussians and the scanned tile counts in that order
// ---------------------------------------------------------------------------------------

constexpr int kOffsetsShare = 16 * kProjBlock; // Gaussians of a workgroup of ordered_offsets_kernel
constexpr int kRanksMax = 131072;              // Gaussians whose depth order is one launch, order_ranks_kernel
constexpr int kBucketBitsMost = 11, kBucketsMost = 4096; // wanted keys of a bucket of depth_scatter_kernel, how many buckets there may be
constexpr int kDepthBinBitsMost = 14;
constexpr size_t kBucketsBytes = ((size_t)4 << kDepthBinBitsMost) + (size_t)kBucketsMost * 8 + 256 + (size_t)(kBucketsMost + 32) * 8 +
                                 (size_t)(kSpanWords + 60 + kSpanChunks) * 4; // (bins, cursors, done, starts, span of BucketsJob)
static_assert(kBucketsBytes % 256 == 0, "whole lines");
static bool orders_by_buckets(int64_t n)
{
    return n > kRanksMax && n <= (int64_t)kBucketsMost << kBucketBitsMost;
}

OrderLayout order_layout(int64_t n, int image_width, int image_height, int list_bin)
{
    auto align = [](size_t x) { return (x + 255) & ~(size_t)255; };
    OrderLayout o;
    size_t off = 0;
    o.depth_keys = off;
    off = align(off + (size_t)n * 4);
    o.ids_a = off;
    off = align(off + (size_t)n * 4);
    o.rects = off;
    off = align(off + (size_t)n * 8);
    o.rects_sorted = off;
    off = align(off + (size_t)n * 8);
    o.records = o.keys_alt = off;
    off = align(off + (size_t)n * 4);
    o.ids_b = off;
    off = align(off + (size_t)n * 4);
    o.rects32 = off;
    off = align(off + (size_t)n * 4);
    if(orders_by_buckets(n))
        off = std::max(off, align(o.records + (size_t)n * 16));
    o.block_sums = off;
    off = align(off + (size_t)((n + kProjBlock - 1) / kProjBlock + 1) * 4);
    o.key_ranges = off;
    off = align(off + (size_t)((n + kProjBlock - 1) / kProjBlock) * 8);
    o.slot_hist = off;
    static_assert(kMaxPasses32 * kBins32 <= 1 << kWideBits, "either");
    off = align(off + ((size_t)1 << kWideBits) * 4);
    o.sort = off;
    off = align(off + sort32_workspace(n, 32, sort32_tile_keys(n)).bytes);
    const ListGrid g = list_grid(image_width, image_height, list_bin);
    o.cover = off;
    off += (size_t)((g.ntx + 1) * (g.nty + 1) + 1) * 4;
    o.bin_cover = off;
    if(g.shift)
        off += (size_t)((g.nbx + 1) * (g.nby + 1) + 1) * 4;
    off = (off + 7) & ~(size_t)7;
    o.key_count = off; // inside the region that is zeroed with the corner grids
    off += 40;
    o.offsets = off; // so is this
    off += 8 * (size_t)((n + kOffsetsShare - 1) / kOffsetsShare);
    o.run_sums = off; // and this
    off = align(off + (n <= kRanksMax ? 4 * (size_t)((n + kProjBlock - 1) / kProjBlock) : 0));
    o.buckets = off; // and this
    off += orders_by_buckets(n) ? kBucketsBytes : 0;
    o.ranges = off;
    off += (size_t)ranges_layout(g).ready * 4;
    o.bytes = align(off);
    return o;
}

__device__ __forceinline__ uint32_t rect_count(uint2 r)
{
    return (r.y & 0xffffu) * ((r.y >> 16) & 0x7fffu);
}

// The bins a tile rectangle touches: first bin (x, y) and extent, for a rectangle that is not empty.
struct BinRect
{
    uint32_t bx, by, bw, bh;
};
__device__ __forceinline__ BinRect bin_rect(uint2 r, int shift)
{
    const uint32_t sx = r.x & 0xffffu, sy = r.x >> 16;
    const uint32_t w = r.y & 0xffffu, h = (r.y >> 16) & 0x7fffu;
    BinRect b;
    b.bx = sx >> shift;
    b.by = sy >> shift;
    b.bw = ((sx + w - 1u) >> shift) - b.bx + 1u;
    b.bh = ((sy + h - 1u) >> shift) - b.by + 1u;
    return b;
}
// Pairs a Gaussian contributes to the lists: one per bin its rectangle touches (shift = 0: one
// per tile).  A Gaussian with a negative depth is in no bin list; its pairs all sit in slot 0,
// as many as the per-tile lists have, so that slot 0 is the same list whatever the bin size.
__device__ __forceinline__ uint32_t list_count(uint2 r, int shift)
{
    const uint32_t fine = rect_count(r);
    if(shift == 0 || fine == 0 || (r.y >> 31))
        return fine;
    const BinRect b = bin_rect(r, shift);
    return b.bw * b.bh;
}

// Where the pairs of each run of 256 Gaussians taken in depth order begin (the last pass of the depth sort
// has already put the rectangles into that order: those of the first `emitting` Gaussians; the others', as far as the
// emission looks at them, are cleared here), and behind them the number of all pairs.
// One launch for the runs' sums and their scan: a workgroup sums up sixteen runs, tells the others, and adds up what those before it
// say.  Bounded by the way of these words from one die to another; us of the two kernels that did it before, a sum and a scan by one
// workgroup -> now: 6 M Gaussians 27.8 -> 18.8, 3 M 16.6 -> 11.6, 1 M 8.5 -> 6.3, 100 K 5.6 -> 5.6.  (64 runs per workgroup: 10.7, 9.5,
// 9.7 and 8.1.)
// A workgroup waits for those before it only.  It takes its number from its place in the grid (one drawn from a counter: 1 us more), so
// whether they run at all is the dispatcher's order: who has waited long enough adds up the other's rectangles itself.
constexpr int kOffsetsThreads = 1024;
constexpr int kOffsetsRuns = kOffsetsShare / kProjBlock; // per workgroup
static_assert(kOffsetsRuns == kOffsetsThreads / DSX_WAVE, "a wavefront for each run");
__global__ __launch_bounds__(kOffsetsThreads) void ordered_offsets_kernel(uint2* __restrict__ rects_sorted, int64_t n,
                                                                          int64_t emitting, int shift,
                                                                          uint32_t* __restrict__ offsets,
                                                                          unsigned long long* __restrict__ state, // a word per workgroup
                                                                          int patience)
{
    constexpr unsigned long long kReady = 1ull << 63;
    __shared__ uint32_t s_sums[kOffsetsRuns];
    __shared__ unsigned long long s_before[kOffsetsThreads / DSX_WAVE];
    const int tid = threadIdx.x, lane = tid & (DSX_WAVE - 1), wave = tid / DSX_WAVE;
    const int64_t share = blockIdx.x, first = share * kOffsetsShare + wave * kProjBlock + lane;
    const int64_t kept = (emitting + kProjBlock - 1) / kProjBlock * kProjBlock; // what the emission looks at
    uint2 r[kProjBlock / DSX_WAVE];
#pragma unroll
    for(int i = 0; i < kProjBlock / DSX_WAVE; ++i)
    {
        const int64_t p = first + i * DSX_WAVE;
        r[i] = make_uint2(0u, 0u);
        if(p < emitting)
            r[i] = rects_sorted[p];
        else if(p < n && p < kept)
            rects_sorted[p] = make_uint2(0u, 0u);
    }
    uint32_t count = 0;
#pragma unroll
    for(int i = 0; i < kProjBlock / DSX_WAVE; ++i)
        count += list_count(r[i], shift);
    count = wave_sum_u32(count);
    if(lane == 0)
        s_sums[wave] = count;
    __syncthreads();
    const uint32_t mine = lane < kOffsetsRuns ? s_sums[lane & (kOffsetsRuns - 1)] : 0u;
    unsigned long long all = mine; // (64 bits: what does not fit 32 is refused by the callers, but must not look like less)
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        all += __shfl_xor(all, o, DSX_WAVE);
    if(tid == 0)
        __hip_atomic_store(state + share, kReady | all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long before = 0;
    for(int64_t b = tid; b < share; b += kOffsetsThreads)
    {
        unsigned long long v = 0;
        for(int spins = 0;; ++spins)
        {
            if(spins > patience)
            {
                v = 0;
                for(int64_t p = b * kOffsetsShare; p < (b + 1) * kOffsetsShare && p < emitting; ++p)
                    v += list_count(rects_sorted[p], shift);
                break;
            }
            v = __hip_atomic_load(state + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if(v & kReady)
                break;
            __builtin_amdgcn_s_sleep(1);
        }
        before += v & ~kReady;
    }
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        before += __shfl_xor(before, o, DSX_WAVE);
    if(lane == 0)
        s_before[wave] = before;
    __syncthreads();
    before = 0;
#pragma unroll
    for(int w = 0; w < kOffsetsThreads / DSX_WAVE; ++w)
        before += s_before[w];
    const int64_t runs = (n + kProjBlock - 1) / kProjBlock, run = share * kOffsetsRuns + lane;
    if(wave == 0)
    {
        const uint32_t incl = wave_incl_scan32(mine, lane);
        if(lane < kOffsetsRuns && run < runs)
            offsets[run] = (uint32_t)before + incl - mine;
        if(share == (runs - 1) / kOffsetsRuns && lane == 0)
        {
            const unsigned long long total = before + all;
            offsets[runs] = total > 0xffffffffull ? 0xffffffffu : (uint32_t)total; // saturates: callers reject counts >= 2^30
        }
    }
}

// ---------------------------------------------------------------------------------------
// 131073 to 8388608 Gaussians: the depth order by buckets, and the block offsets with it
// ---------------------------------------------------------------------------------------
// Two launches behind a histogram of 2^12 to 2^14 bins of the depths' range.  A bucket is the bins whose middle lies in 1024 or 2048
// consecutive ranks (a bin of more keys than that is then nearly all of its bucket), so its first rank is known, and a workgroup of the
// first launch needs no other's ranks: it counts its keys by bucket in LDS, asks for that much room in each (one atomic per bucket and
// workgroup) and writes (key, index, rectangle) there, in any order.  The second launch sorts a bucket at a time in LDS (4096 bins of its
// own range of (key, index), the few in the same bin compared with each other) and writes order and rectangles; the pairs of a bucket
// were summed with its room, so the block offsets fall out as well.
// Nobody waits for another workgroup.
// Where a bucket would have more keys than it has room for, because a bin of the range holds thousands (many equal depths, or most
// of a cloud in a small part of a wide range), the first launch counts the digits of the passes instead, which run then; where the range
// has both signs, or is wide or thin, the host sees that beforehand.  us of a forward at 1280x720 with the passes alone -> now: nine
// tenths of the depths within 0.7 of twelve octaves 200 K 209 -> 187, 600 K 281 -> 273, 1 M 339 -> 345 (too full), 3 M 617 -> 614 (too
// full); two depths 140 K 167 -> 170, 300 K 236 -> 232, 1 M 343 -> 343, 2 M 468 -> 472, 3 M 625 -> 630.  (With the histogram of the
// digits in another launch and a clear before it: two depths 195, 258, 366, 3 M 664.)
// The first launch is bound by latency (ranges and bins 4 us, the table 3, keys and rectangles 4, room 2, the stores 3 to 10: two rounds
// of workgroups beyond 3 M) and by its scattered stores, whose partial lines are 69 MB instead of 34 for 3 M (2 M of them emitting); the
// second by its chain of short steps, four workgroups at a time on a compute unit.  us alone: 300 K 11 + 8, 500 K 14 + 9, 1 M 20 + 14,
// 3 M 38 + 21, 6 M 77 + 34; the digit passes and the offsets were 42, 47, 57, 97 and 182.  A whole forward, 1280x720, of 150 K Gaussians
// 120 -> 100 us, 250 K 144 -> 117, 600 K 195 -> 173, 1.5 M 263 -> 240, 4 M 422 -> 384; a training step of 3 M at 1920x1080 752 -> 710.
// (Tried: buckets of 1024 and workgroups of 8192 keys, whose two records a bucket and workgroup are nearly all partial lines: 65 us at
// 3 M; no keys in registers but read twice, by twice the workgroups: 46; buckets of 4096, whose sort takes 27 instead of 21.)
constexpr int kScatterThreads = 1024;
constexpr int kScatterWaves = kScatterThreads / DSX_WAVE;
constexpr int kBucketThreads = 512;
constexpr int kBucketWaves = kBucketThreads / DSX_WAVE;
constexpr int kBucketItems = 8;
constexpr int kBucketKeys = 4032; // that a bucket can have (as many as let four workgroups share a compute unit's LDS)
constexpr int kBucketBinBits = 12;
constexpr uint32_t kBucketGroupMost = 64; // keys in one bin that are compared with each other one by one
constexpr uint64_t kBucketsDone = 1, kBucketsTooFull = 2;
constexpr int kPairsAt = 24; // bits of a rank
static_assert(((int64_t)kBucketsMost << kBucketBitsMost) <= 1 << kPairsAt, "ranks");

struct BucketsJob
{
    const uint32_t* keys; // by Gaussian
    const uint2* rects;
    const uint2* key_ranges; // of 256 consecutive Gaussians (see OrderLayout)
    uint32_t* bins;              // (zero at first)
    uint32_t* digits;            // histograms of the passes' digits, where the buckets cannot be had (zero at first)
    uint32_t* span;              // (see depth_hist_kernel)
    unsigned long long* cursors; // of each bucket: keys, and their pairs << kPairsAt (zero at first)
    uint2* starts;               // of each bucket and behind the last: its first rank, the pairs before it
    uint32_t* done;              // workgroups that have asked for their room; whether there are starts (both zero at first)
    Words4* records;
    uint32_t* order; // by depth
    uint2* rects_sorted;
    uint32_t* block_sums;
    int n, shift, buckets, bucket_bits;
    HostCounts to_host;
};

// kRuns: of 256 Gaussians, of a wavefront, whose keys and rectangles stay in its registers
template <int kRuns, int kBinBits>
__global__ __launch_bounds__(kScatterThreads) void depth_scatter_kernel(const BucketsJob J)
{
    constexpr int kBins = 1 << kBinBits, kMine = kBins / kScatterThreads, kEach = kBucketsMost / kScatterThreads;
    constexpr int kParts = kProjBlock / DSX_WAVE;
    extern __shared__ __attribute__((aligned(16))) unsigned long long s_taken[]; // this workgroup's keys of the bucket, their pairs << kPairsAt
    uint32_t* const s_room = reinterpret_cast<uint32_t*>(s_taken + kBucketsMost); // the bucket's first rank, then where its next key goes
    uint16_t* const s_bucket = reinterpret_cast<uint16_t*>(s_room + kBucketsMost); // of each bin
    __shared__ uint32_t s_emit[kRuns * kScatterWaves];   // of each of this workgroup's runs: emitting Gaussians before it
    __shared__ __attribute__((aligned(16))) uint32_t s_tot[kScatterWaves];
    __shared__ uint2 s_part[kScatterWaves];
    __shared__ unsigned long long s_all[kScatterWaves];
    __shared__ uint32_t s_flag, s_front;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = J.n, blocks = (n + kProjBlock - 1) / kProjBlock;
    const int run0 = (int)blockIdx.x * (kRuns * kScatterWaves);
    auto index_of = [&](int q, int u) { return (run0 + q * kScatterWaves + wave) * kProjBlock + u * DSX_WAVE + lane; };

    Words4 bin4[kMine / 4];
#pragma unroll
    for(int q = 0; q < kMine / 4; ++q)
        bin4[q] = reinterpret_cast<const Words4*>(J.bins)[(kMine / 4) * tid + q];
    uint32_t key[kRuns][kParts];
#pragma unroll
    for(int q = 0; q < kRuns; ++q)
#pragma unroll
        for(int u = 0; u < kParts; ++u)
            key[q][u] = index_of(q, u) < n ? J.keys[index_of(q, u)] : kNoPairsKey;
    const int chunk = span_chunk(blocks), front = run0 / chunk;
    const uint32_t emitting = J.span[2], front_emits = J.span[kSpanWords + front];
    const DepthRange range = depth_range(0xffffu - J.span[0], J.span[1]);
    // (fewer runs than a wavefront has lanes lie between a chunk's first one and this workgroup's)
    const uint32_t between = wave == 0 && front * chunk + lane < run0 ? J.key_ranges[front * chunk + lane].x >> 16 : 0u;
    const uint32_t run_emits = tid < kRuns * kScatterWaves && run0 + tid < blocks ? J.key_ranges[run0 + tid].x >> 16 : 0u;
    static_assert(((int64_t)kBucketsMost << kBucketBitsMost) / kProjBlock / kSpanChunks <= DSX_WAVE, "a lane for each");
    uint32_t sum = 0, most = 0;
#pragma unroll
    for(int q = 0; q < kMine / 4; ++q)
    {
        sum += bin4[q].x + bin4[q].y + bin4[q].z + bin4[q].w;
        most = max(max(max(most, bin4[q].x), max(bin4[q].y, bin4[q].z)), bin4[q].w);
    }
    const uint32_t incl = wave_incl_scan_u32(sum), runs_incl = wave_incl_scan_u32(run_emits), between_all = wave_sum_u32(between);
    if(lane == 63)
    {
        s_tot[wave] = incl;
        s_part[wave].x = runs_incl;
    }
    if(tid == 0)
    {
        s_flag = 0;
        s_front = front_emits + between_all;
    }
#pragma unroll
    for(int q = 0; q < kEach; ++q)
    {
        s_room[q * kScatterThreads + tid] = 0xffffffffu;
        s_taken[q * kScatterThreads + tid] = 0;
    }
    __syncthreads();
    if(tid < kRuns * kScatterWaves)
        s_emit[tid] = s_front + (wave ? s_part[0].x : 0u) + runs_incl - run_emits;
    static_assert(kRuns * kScatterWaves <= 2 * DSX_WAVE, "two wavefronts' runs");
    const uint32_t at_first = sum_of_waves_before<kScatterWaves>(s_tot, wave) + incl - sum;
    uint32_t at = at_first, last_bucket = 0xffffffffu;
#pragma unroll
    for(int q = 0; q < kMine / 4; ++q)
    {
        const uint32_t count[4] = {bin4[q].x, bin4[q].y, bin4[q].z, bin4[q].w};
        uint32_t bucket[4];
#pragma unroll
        for(int u = 0; u < 4; ++u)
        {
            bucket[u] = min((at + count[u] / 2) >> J.bucket_bits, (uint32_t)J.buckets - 1u);
            if(count[u] && bucket[u] != last_bucket)
            {
                atomicMin(&s_room[bucket[u]], at);
                last_bucket = bucket[u];
            }
            at += count[u];
        }
        *reinterpret_cast<uint2*>(s_bucket + kMine * tid + 4 * q) = make_uint2(bucket[0] | bucket[1] << 16, bucket[2] | bucket[3] << 16);
    }
    if(most > kBucketKeys - (1u << J.bucket_bits))
        atomicMax(&s_flag, most);
    uint2 rect[kRuns][kParts];
#pragma unroll
    for(int q = 0; q < kRuns; ++q)
#pragma unroll
        for(int u = 0; u < kParts; ++u)
            rect[q][u] = key[q][u] != kNoPairsKey ? J.rects[index_of(q, u)] : make_uint2(0u, 0u);
    __syncthreads();
    const uint32_t fullest = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_flag); // (of the bins, if a bucket may be too full for it)
    bool too_full = fullest > (uint32_t)kBucketKeys;
    if(fullest != 0 && !too_full)
    {
        // has one?
        uint32_t end = at_first;
        bool over = false;
#pragma unroll
        for(int q = 0; q < kMine / 4; ++q)
        {
            const Words4 four = reinterpret_cast<const Words4*>(J.bins)[(kMine / 4) * tid + q];
            const uint32_t count[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
            for(int u = 0; u < 4; ++u)
            {
                const uint32_t first = s_room[s_bucket[kMine * tid + 4 * q + u]]; // (of an empty bin's bucket perhaps none)
                end += count[u];
                over |= count[u] != 0 && end - first > (uint32_t)kBucketKeys;
            }
        }
        __syncthreads();
        if(tid == 0)
            s_flag = 0;
        __syncthreads();
        if(over)
            s_flag = 1;
        __syncthreads();
        too_full = __builtin_amdgcn_readfirstlane((int)s_flag) != 0;
    }
    if(blockIdx.x == 0 && tid == 0)
        store_to_host(J.to_host, 4, too_full ? kBucketsTooFull : kBucketsDone);
    if(too_full) // (every workgroup finds so)
    {
        // the digits of this workgroup's keys, for the passes, which come next
        uint32_t* const s_digits = reinterpret_cast<uint32_t*>(s_taken);
        static_assert(kDepthPasses * kDepthBins <= 2 * kBucketsMost, "room");
        auto count_digits = [&](auto crowded) {
#pragma unroll
            for(int q = 0; q < kRuns; ++q)
#pragma unroll
                for(int u = 0; u < kParts; ++u)
#pragma unroll
                    for(int p = 0; p < kDepthPasses; ++p)
                    {
                        const uint32_t digit = ((key[q][u] - range.first) >> range.digits.shift[p]) & range.digits.mask[p];
                        bool todo = key[q][u] != kNoPairsKey;
                        if(decltype(crowded)::value)
#pragma unroll
                            for(int r = 0; r < 2; ++r)
                            {
                                const uint64_t left = __builtin_amdgcn_ballot_w64(todo);
                                const int leader = left ? __builtin_ctzll(left) : 0;
                                const bool same = todo && digit == (uint32_t)__builtin_amdgcn_readlane((int)digit, leader);
                                const uint64_t alike = __builtin_amdgcn_ballot_w64(same);
                                if(lane == leader && same)
                                    atomicAdd(&s_digits[p * kDepthBins + digit], (uint32_t)__popcll(alike));
                                todo = todo && !same;
                            }
                        if(todo)
                            atomicAdd(&s_digits[p * kDepthBins + digit], 1u);
                    }
        };
        // (additions to one word go one by one: where a bin holds many, two of a wavefront's digits are added up first.  us of a forward
        // of 3 M at two depths 648 -> 626, at depths of which nine tenths lie within 0.7 of twelve octaves, if it were done there, 621
        // -> 627)
        if(fullest > emitting / 32)
            count_digits(std::true_type());
        else
            count_digits(std::false_type());
        __syncthreads();
        for(int j = tid; j < kDepthPasses * kDepthBins; j += kScatterThreads)
            if(s_digits[j])
                atomicAdd(&J.digits[j], s_digits[j]);
        return;
    }
    const uint32_t scale = depth_bin_scale(range, kBinBits);
    auto bucket_of = [&](uint32_t k) { return s_bucket[min(depth_bin(k - range.first, scale), (uint32_t)(kBins - 1))]; };
#pragma unroll
    for(int q = 0; q < kRuns; ++q)
#pragma unroll
        for(int u = 0; u < kParts; ++u)
            if(key[q][u] != kNoPairsKey) // (what a wide rectangle counts is cut off where the callers refuse the sum)
                atomicAdd(&s_taken[bucket_of(key[q][u])],
                          (unsigned long long)min(list_count(rect[q][u], J.shift), 1u << 30) << kPairsAt | 1ull);
    __syncthreads();
    uint32_t back[kEach];
#pragma unroll
    for(int q = 0; q < kEach; ++q)
    {
        const int b = q * kScatterThreads + tid;
        const unsigned long long mine = s_taken[b];
        back[q] = 0;
        if(mine)
            back[q] = (uint32_t)atomicAdd(&J.cursors[b], mine) & ((1u << kPairsAt) - 1u);
    }
#pragma unroll
    for(int q = 0; q < kEach; ++q) // (an addition has been performed when its result is back)
        s_room[q * kScatterThreads + tid] += back[q];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if(tid == 0)
        s_flag = atomicAdd(J.done, 1u) == gridDim.x - 1;
    const uint32_t kept = (emitting + kProjBlock - 1) / kProjBlock * kProjBlock; // what the emission looks at
#pragma unroll
    for(int q = 0; q < kRuns; ++q)
    {
        // (those that emit nothing: behind the others, by index)
        uint32_t behind = emitting + (uint32_t)((run0 + q * kScatterWaves + wave) * kProjBlock) - s_emit[q * kScatterWaves + wave];
#pragma unroll
        for(int u = 0; u < kParts; ++u)
        {
            const uint32_t i = (uint32_t)index_of(q, u);
            const uint64_t none = __builtin_amdgcn_ballot_w64(key[q][u] == kNoPairsKey);
            if(key[q][u] != kNoPairsKey)
            {
                const uint32_t p = atomicAdd(&s_room[bucket_of(key[q][u])], 1u);
                J.records[min(p, (uint32_t)n - 1u)] = Words4{key[q][u], i, rect[q][u].x, rect[q][u].y};
            }
            else if(i < (uint32_t)n)
            {
                const uint32_t p = min(behind + bits_below(none), (uint32_t)n - 1u);
                J.order[p] = i;
                if(p < kept)
                    J.rects_sorted[p] = make_uint2(0u, 0u);
            }
            behind += (uint32_t)__popcll(none);
        }
    }
    __syncthreads();
    // the last workgroup sums the buckets up
    if(!s_flag)
        return;
    uint32_t keys[kEach], own_keys = 0, own_pairs = 0;
    unsigned long long pairs[kEach], all = 0;
#pragma unroll
    for(int q = 0; q < kEach; ++q)
    {
        const unsigned long long taken = __hip_atomic_load(J.cursors + kEach * tid + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        keys[q] = (uint32_t)taken & ((1u << kPairsAt) - 1u);
        pairs[q] = taken >> kPairsAt;
    }
#pragma unroll
    for(int q = 0; q < kEach; ++q)
    {
        own_keys += keys[q];
        own_pairs += (uint32_t)pairs[q];
        all += pairs[q]; // (64 bits: what does not fit 32 is refused by the callers, but must not look like less)
    }
    const uint32_t keys_incl = wave_incl_scan_u32(own_keys), pairs_incl = wave_incl_scan_u32(own_pairs);
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        all += __shfl_xor(all, o, DSX_WAVE);
    if(lane == 63)
    {
        s_part[wave] = make_uint2(keys_incl, pairs_incl);
        s_all[wave] = all;
    }
    __syncthreads();
    uint32_t rank = keys_incl - own_keys, before = pairs_incl - own_pairs;
    all = 0;
#pragma unroll
    for(int w = 0; w < kScatterWaves; ++w)
    {
        rank += w < wave ? s_part[w].x : 0u;
        before += w < wave ? s_part[w].y : 0u;
        all += s_all[w];
    }
#pragma unroll
    for(int q = 0; q < kEach; ++q)
    {
        J.starts[kEach * tid + q] = make_uint2(rank, before);
        rank += keys[q];
        before += (uint32_t)pairs[q];
    }
    const uint32_t total = all > 0xffffffffull ? 0xffffffffu : (uint32_t)all;
    for(int run = (int)(kept / kProjBlock) + tid; run <= blocks; run += kScatterThreads)
        J.block_sums[run] = total;
    if(tid == 0)
    {
        J.starts[kBucketsMost] = make_uint2(emitting, total);
        J.done[1] = 1u;
    }
}

// (39 KB of LDS and 64 registers: four workgroups to a compute unit)
__global__ __launch_bounds__(kBucketThreads) __attribute__((amdgpu_waves_per_eu(8))) void order_buckets_kernel(const BucketsJob J)
{
    constexpr int kBins = 1 << kBucketBinBits;
    __shared__ __attribute__((aligned(16))) uint64_t s_binned[kBucketKeys];
    __shared__ __attribute__((aligned(16))) uint16_t s_hist[kBins]; // two in a word
    __shared__ __attribute__((aligned(16))) uint32_t s_tot[kBucketWaves];
    __shared__ uint2 s_ends[kBucketWaves];
    __shared__ uint32_t s_sums[kBucketKeys / kProjBlock + 2];
    __shared__ uint32_t s_alike;
    uint32_t* const s_pairs = reinterpret_cast<uint32_t*>(s_hist);
    static_assert(kBins == 8 * kBucketThreads && kBucketKeys <= kBucketItems * kBucketThreads && kBucketKeys <= kBins, "what the threads take");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint2 start = J.starts[blockIdx.x];
    const int count = J.done[1] ? (int)min(J.starts[blockIdx.x + 1].x - start.x, (uint32_t)kBucketKeys) : 0;
    if(count == 0) // (uniform)
        return;
    uint64_t mine[kBucketItems]; // key, index
    uint2 rect[kBucketItems];
    uint32_t nearest = 0, farthest = 0; // (the former's complement)
#pragma unroll
    for(int it = 0; it < kBucketItems; ++it)
    {
        const int at = it * kBucketThreads + tid;
        mine[it] = ~0ull;
        rect[it] = make_uint2(0u, 0u);
        if(at < count)
        {
            const Words4 record = J.records[start.x + at];
            mine[it] = (uint64_t)record.x << 32 | record.y;
            rect[it] = make_uint2(record.z, record.w);
            nearest = max(nearest, ~record.x);
            farthest = max(farthest, record.x);
        }
    }
    nearest = wave_incl_max_scan(nearest);
    farthest = wave_incl_max_scan(farthest);
    if(lane == 63)
        s_ends[wave] = make_uint2(nearest, farthest);
    reinterpret_cast<uint4*>(s_hist)[tid] = make_uint4(0u, 0u, 0u, 0u);
    if(tid < kBucketKeys / kProjBlock + 2)
        s_sums[tid] = 0;
    if(tid == 0)
        s_alike = 0;
    __syncthreads();
    nearest = farthest = 0;
#pragma unroll
    for(int w = 0; w < kBucketWaves; ++w)
    {
        nearest = max(nearest, s_ends[w].x);
        farthest = max(farthest, s_ends[w].y);
    }
    nearest = ~(uint32_t)__builtin_amdgcn_readfirstlane((int)nearest);
    farthest = (uint32_t)__builtin_amdgcn_readfirstlane((int)farthest);
    const uint64_t from = (uint64_t)nearest << 32;
    const int to_bin = (farthest == nearest ? 32 : 64 - __builtin_clz(farthest - nearest)) - kBucketBinBits;
    uint32_t place[kBucketItems]; // bin << 16 | how many came before; then the bin's first place, the one behind its last << 16
    uint32_t most = 0;
#pragma unroll
    for(int it = 0; it < kBucketItems; ++it)
    {
        place[it] = 0;
        if(it * kBucketThreads + tid < count)
        {
            const uint32_t bin = (uint32_t)((mine[it] - from) >> to_bin), half = 16 * (bin & 1);
            const uint32_t nth = atomicAdd(&s_pairs[bin >> 1], 1u << half) >> half & 0xffffu;
            place[it] = bin << 16 | nth;
            most = max(most, nth);
        }
    }
    if(__builtin_amdgcn_ballot_w64(most >= kBucketGroupMost) != 0 && lane == 0)
        s_alike = 1;
    __syncthreads();
    // exclusive sums of the bins
    {
        uint4* const eight = reinterpret_cast<uint4*>(s_hist) + tid;
        const uint4 c = *eight;
        const uint32_t both = c.x + c.y + c.z + c.w, sum = (both & 0xffffu) + (both >> 16), incl = wave_incl_scan_u32(sum);
        if(lane == 63)
            s_tot[wave] = incl;
        __syncthreads();
        uint32_t at = sum_of_waves_before<kBucketWaves>(s_tot, wave) + incl - sum;
        auto two = [&](uint32_t w) {
            const uint32_t first = at, second = at + (w & 0xffffu);
            at = second + (w >> 16);
            return first | second << 16;
        };
        const uint32_t x = two(c.x), y = two(c.y), z = two(c.z), w = two(c.w);
        *eight = make_uint4(x, y, z, w);
    }
    __syncthreads();
    const bool alike = __builtin_amdgcn_readfirstlane((int)s_alike) != 0;
    uint32_t rank[kBucketItems];
    if(!alike)
    {
        uint32_t longest = 0;
#pragma unroll
        for(int it = 0; it < kBucketItems; ++it)
        {
            rank[it] = 0;
            if(it * kBucketThreads + tid < count)
            {
                const uint32_t bin = place[it] >> 16, first = s_hist[bin];
                const uint32_t end = bin + 1 < (uint32_t)kBins ? s_hist[bin + 1] : (uint32_t)count;
                s_binned[first + (place[it] & 0xffffu)] = mine[it];
                place[it] = first | end << 16;
                rank[it] = first;
                longest = max(longest, end - first);
            }
        }
        __syncthreads();
        for(uint32_t j = 0; __builtin_amdgcn_ballot_w64(j < longest) != 0; ++j)
#pragma unroll
            for(int it = 0; it < kBucketItems; ++it)
                if((place[it] & 0xffffu) + j < place[it] >> 16)
                    rank[it] += s_binned[(place[it] & 0xffffu) + j] < mine[it] ? 1u : 0u;
    }
    else
    {
        // many depths alike: a bitonic sort, and everybody looks for its own
        // (the steps are those of the next power of two; what would lie behind the last key is larger than all)
        int size = kBucketThreads;
        while(size < count)
            size *= 2;
#pragma unroll
        for(int it = 0; it < kBucketItems; ++it)
            if(it * kBucketThreads + tid < count)
                s_binned[it * kBucketThreads + tid] = mine[it];
        for(int k = 2; k <= size; k *= 2)
            for(int j = k / 2; j > 0; j /= 2)
            {
                __syncthreads();
                for(int e = tid; e < size / 2; e += kBucketThreads)
                {
                    // (the first step of each size mirrors its second half: the smaller always comes first)
                    const int i = 2 * e - (e & (j - 1)), l = j == k / 2 ? i + (k - 1 - 2 * (i & (k - 1))) : i + j;
                    if(l >= count)
                        continue;
                    const uint64_t u = s_binned[i], v = s_binned[l];
                    if(u > v)
                    {
                        s_binned[i] = v;
                        s_binned[l] = u;
                    }
                }
            }
        __syncthreads();
#pragma unroll
        for(int it = 0; it < kBucketItems; ++it)
        {
            uint32_t r = 0;
            if(it * kBucketThreads + tid < count)
                for(int step = size / 2; step > 0; step /= 2)
                    if(r + step <= (uint32_t)count && s_binned[r + step - 1] < mine[it])
                        r += step;
            rank[it] = r;
        }
    }
    __syncthreads();
    // the rectangles in order, the runs' sums, and the order
    uint2* const s_rects = reinterpret_cast<uint2*>(s_binned);
    uint32_t* const s_ids = reinterpret_cast<uint32_t*>(s_binned);
#pragma unroll
    for(int it = 0; it < kBucketItems; ++it)
        if(it * kBucketThreads + tid < count)
            s_rects[rank[it]] = rect[it];
    __syncthreads();
    const uint32_t run0 = start.x / kProjBlock;
#pragma unroll
    for(int it = 0; it < kBucketItems; ++it)
    {
        if(it * kBucketThreads >= count) // (uniform)
            break;
        const int at = it * kBucketThreads + tid;
        const uint32_t p = start.x + (uint32_t)at;
        uint32_t pairs = 0;
        if(at < count)
        {
            const uint2 r = s_rects[at];
            J.rects_sorted[p] = r;
            pairs = list_count(r, J.shift);
        }
        const uint32_t run = p / kProjBlock - run0, other = (uint32_t)__builtin_amdgcn_readlane((int)run, 63);
        if(__builtin_amdgcn_readfirstlane(run) == other)
        {
            const uint32_t sum = wave_sum_u32(pairs);
            if(lane == 0 && sum)
                atomicAdd(&s_sums[run], sum);
        }
        else if(pairs)
            atomicAdd(&s_sums[run], pairs);
    }
    __syncthreads();
#pragma unroll
    for(int it = 0; it < kBucketItems; ++it)
        if(it * kBucketThreads + tid < count)
            s_ids[rank[it]] = (uint32_t)mine[it];
    __syncthreads();
    for(int at = tid; at < count; at += kBucketThreads)
        J.order[start.x + at] = s_ids[at];
    // (of the runs that begin here)
    static_assert(kBucketKeys / kProjBlock + 2 <= DSX_WAVE, "a lane for each run");
    if(wave == 0)
    {
        const uint32_t sum = lane < kBucketKeys / kProjBlock + 2 ? s_sums[lane] : 0u, before = start.y + wave_incl_scan_u32(sum) - sum;
        const uint32_t p = (run0 + (uint32_t)lane) * kProjBlock;
        if(p >= start.x && p < start.x + (uint32_t)count)
            J.block_sums[run0 + lane] = before;
    }
}

// How many pairs each tile receives, straight from the rectangles (no pair is enumerated):
// a rectangle [sx, ex) x [sy, ey) adds +1, -1, -1, +1 at its four corners of a
// (nty + 1) x (ntx + 1) grid, and the two-dimensional prefix sum of that grid is the number of
// rectangles covering each tile.  Pairs of a Gaussian with a negative depth all sit in slot 0:
// they are counted in the cell after the grid.  From the per-tile counts come the digit
// histograms of the tile partition (and the tile counts themselves).
constexpr int kCoverThreads = 1024;
constexpr int kCoverBlocks = 128;
constexpr int kCoverLdsCells = 14 * 1024;      // grids up to this many cells (56 KB) are held in LDS as they are
constexpr int kCoverLdsCellsLarge = 38 * 1024; // up to 152 KB of the CU's 160 KB, once the kernels are allowed it

// shift > 0: the same for the bins, into a second grid right behind the first (bin_grid); the
// pairs of the bin lists are summed into key_count[1].
__global__ __launch_bounds__(kCoverThreads) void tile_cover_kernel(const uint2* __restrict__ rects, int64_t n, int ntx,
                                                                   int nty, int shift, int nbx, int nby, int use_lds,
                                                                   int32_t* __restrict__ grid,
                                                                   int32_t* __restrict__ bin_grid,
                                                                   unsigned long long* __restrict__ key_count,
                                                                   const HostCounts to_host)
{
    extern __shared__ int32_t s_grid[];
    const int tid = threadIdx.x;
    unsigned long long pairs = 0;     // tiles of this thread's rectangles: summed over the launch this is K
    unsigned long long bin_pairs = 0; // the same for the bin lists
    const int pitch = ntx + 1;
    const int cells = pitch * (nty + 1) + 1;
    const int bpitch = nbx + 1;
    const int bcells = shift ? bpitch * (nby + 1) + 1 : 0;
    int32_t* acc = use_lds ? s_grid : grid;
    int32_t* bacc = use_lds ? s_grid + cells : bin_grid;
    if(use_lds)
    {
        for(int j = tid; j < cells + bcells; j += kCoverThreads)
            s_grid[j] = 0;
        __syncthreads();
    }
    constexpr int kAhead = 4; // rectangles whose loads are in flight
    const int64_t stride = (int64_t)gridDim.x * kCoverThreads;
    for(int64_t g0 = (int64_t)blockIdx.x * kCoverThreads + tid; g0 < n; g0 += kAhead * stride)
    {
        uint2 ahead[kAhead];
#pragma unroll
        for(int u = 0; u < kAhead; ++u)
            ahead[u] = g0 + u * stride < n ? rects[g0 + u * stride] : make_uint2(0u, 0u);
#pragma unroll
        for(int u = 0; u < kAhead; ++u)
        {
            const uint2 r = ahead[u];
            const int w = (int)(r.y & 0xffffu), h = (int)((r.y >> 16) & 0x7fffu);
            if(w == 0 || h == 0)
                continue;
            pairs += (unsigned long long)(w * h);
            if(r.y >> 31)
            {
                atomicAdd(&acc[cells - 1], w * h);
                if(shift)
                {
                    atomicAdd(&bacc[bcells - 1], w * h);
                    bin_pairs += (unsigned long long)(w * h);
                }
                continue;
            }
            const int sx = (int)(r.x & 0xffffu), sy = (int)(r.x >> 16);
            atomicAdd(&acc[sy * pitch + sx], 1);
            atomicAdd(&acc[sy * pitch + sx + w], -1);
            atomicAdd(&acc[(sy + h) * pitch + sx], -1);
            atomicAdd(&acc[(sy + h) * pitch + sx + w], 1);
            if(shift)
            {
                const BinRect b = bin_rect(r, shift);
                bin_pairs += (unsigned long long)(b.bw * b.bh);
                atomicAdd(&bacc[b.by * bpitch + b.bx], 1);
                atomicAdd(&bacc[b.by * bpitch + b.bx + b.bw], -1);
                atomicAdd(&bacc[(b.by + b.bh) * bpitch + b.bx], -1);
                atomicAdd(&bacc[(b.by + b.bh) * bpitch + b.bx + b.bw], 1);
            }
        }
    }
    if(use_lds)
    {
        __syncthreads();
        for(int j = tid; j < cells; j += kCoverThreads)
            if(s_grid[j])
                atomicAdd(&grid[j], s_grid[j]);
        for(int j = tid; j < bcells; j += kCoverThreads)
            if(s_grid[cells + j])
                atomicAdd(&bin_grid[j], s_grid[cells + j]);
    }
    // the number of pairs of the whole scene (64 bits: it is compared with the 2^30 limit, not wrapped)
    // (one atomic per workgroup: atomics on one address serialise in the L2)
    __shared__ unsigned long long s_pairs[2][kCoverThreads / DSX_WAVE];
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
    {
        pairs += __shfl_xor(pairs, o, DSX_WAVE);
        bin_pairs += __shfl_xor(bin_pairs, o, DSX_WAVE);
    }
    if((tid & 63) == 0)
    {
        s_pairs[0][tid >> 6] = pairs;
        s_pairs[1][tid >> 6] = bin_pairs;
    }
    __syncthreads();
    if(tid == 0)
    {
        unsigned long long total[2] = {0, 0};
        for(int w = 0; w < kCoverThreads / DSX_WAVE; ++w)
        {
            total[0] += s_pairs[0][w];
            total[1] += s_pairs[1][w];
        }
        // The workgroup that is last to add its sums hands them to the waiting host.  The additions have been
        // performed when their results are back, so the ticket is drawn after them.
        const unsigned long long before0 = atomicAdd(key_count, total[0]), before1 = atomicAdd(key_count + 1, total[1]);
        asm volatile("s_waitcnt vmcnt(0)" ::"v"(before0), "v"(before1) : "memory");
        if(to_host.words && atomicAdd(key_count + 2, 1ull) == gridDim.x - 1)
            for(int i = 0; i < 2; ++i)
                store_to_host(to_host, i, atomicAdd(key_count + i, 0ull));
    }
}

// One workgroup: 2-D prefix sum of the corner grid (in LDS when the grid fits, else in place in
// global memory, where a few ten thousand cells stay in the L2), then
//  * the digit histograms of slot = tile + 1 (slot 0 = the negative depths),
//  * ranges[j] = number of pairs whose tile is below j, with the two rules of the reference
//    (cpp/rasterizer_kernels.cu:313-322, cpp/rasterizer_torch.cu:31-39): the boundary after
//    the LAST run is never recorded, so tiles above the highest occupied tile inherit the
//    START of that run (all zero when no tile is occupied), and ranges[num_tiles] = K.
// Binned lists: workgroup 0 does the above for the tiles (no histograms: nothing is partitioned by
// tile then) and also records the highest occupied tile; workgroup 1 takes the bins' grid, whose
// ranges are plain prefix sums (the reference's two rules are rules about tiles) and whose
// histograms drive the partition.
struct CountsJob
{
    int32_t* grid;
    int ntx, nty;
    int plain;           // 1: ranges are plain prefix sums, no rule about the last run
    uint32_t* slot_hist; // may be null
    int32_t* ranges;
    int32_t* last;       // may be null: receives the highest occupied tile, -1 if none
    int32_t* header;     // may be null: receives header_value (the bin shift the lists are built for)
    int32_t header_value;
    Digits32 plan;
};
struct CountsJobs
{
    CountsJob job[2];
};

// (rounds through the tiles between two barriers; one: the kernel of 2 K Gaussians at 3840x2160 37.6 us, four 36.3)
constexpr int kTileRounds = 4;

// c: the corner grid, wherever it lies (a workgroup's own copy in LDS, or global memory)
__device__ __forceinline__ void tile_counts(const CountsJob& J, int32_t* const c)
{
    const int ntx = J.ntx, nty = J.nty;
    const Digits32& plan = J.plan;
    // one wide digit: a list's pairs are its own bin's, stored as they are counted
    uint32_t* const wide_hist = J.plan.mask[0] >= (uint32_t)kBins32 ? J.slot_hist : nullptr;
    uint32_t* const slot_hist = wide_hist ? nullptr : J.slot_hist;
    int32_t* const ranges = J.ranges;
    __shared__ uint32_t hist[kMaxPasses32 * kBins32];
    __shared__ __attribute__((aligned(16))) uint32_t wave_tot[kTileRounds][kCoverThreads / DSX_WAVE];
    __shared__ int s_last;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int pitch = ntx + 1;
    const int cells = pitch * (nty + 1) + 1;
    const uint32_t negatives = (uint32_t)c[cells - 1];
    for(int j = tid; j < kMaxPasses32 * kBins32; j += kCoverThreads)
        hist[j] = 0;
    if(tid == 0)
        s_last = -1;
    __threadfence_block();
    __syncthreads();
    // along x: one wavefront per row, 64 columns at a time with a carry
    for(int y = wave; y < nty; y += kCoverThreads / DSX_WAVE)
    {
        int32_t carry = 0;
        for(int x0 = 0; x0 < ntx; x0 += DSX_WAVE)
        {
            const int x = x0 + lane;
            const int32_t v = x < ntx ? c[y * pitch + x] : 0;
            const int32_t incl = (int32_t)wave_incl_scan32((uint32_t)v, lane) + carry;
            if(x < ntx)
                c[y * pitch + x] = incl;
            carry = __shfl(incl, 63, DSX_WAVE);
        }
    }
    __threadfence_block();
    __syncthreads();
    // along y: one thread per column
    for(int x = tid; x < ntx; x += kCoverThreads)
    {
        int32_t run = 0;
        for(int y = 0; y < nty; ++y)
        {
            run += c[y * pitch + x];
            c[y * pitch + x] = run; // pairs of tile (x, y)
        }
    }
    __threadfence_block();
    __syncthreads();
    // histograms, exclusive scan over the tiles in row-major order, highest occupied tile
    // (four rounds between two barriers)
    const int tiles = ntx * nty;
    uint32_t carry = negatives;
    for(int t0 = 0; t0 < tiles; t0 += kTileRounds * kCoverThreads)
    {
        uint32_t cnt[kTileRounds], incl[kTileRounds];
#pragma unroll
        for(int u = 0; u < kTileRounds; ++u)
        {
            const int t = t0 + u * kCoverThreads + tid;
            cnt[u] = t < tiles ? (uint32_t)c[(t / ntx) * pitch + (t % ntx)] : 0u;
        }
#pragma unroll
        for(int u = 0; u < kTileRounds; ++u)
        {
            if(t0 + u * kCoverThreads >= tiles) // (uniform)
                break;
            // lanes hold consecutive tiles: the lowest digit differs from lane to lane (plain LDS
            // atomics, no conflicts), a higher digit is constant over long runs (one add per run,
            // after a wavefront sum; same-address LDS atomics would serialise)
            const uint32_t slot = (uint32_t)(t0 + u * kCoverThreads + tid) + 1u;
            if(wide_hist && slot <= plan.mask[0])
                wide_hist[slot] = cnt[u]; // (zero behind the last list)
            for(int p = 0; slot_hist && p < plan.passes; ++p)
            {
                const uint32_t d = (slot >> plan.shift[p]) & plan.mask[p];
                if(plan.shift[p] == 0)
                {
                    if(cnt[u])
                        atomicAdd(&hist[p * kBins32 + d], cnt[u]);
                    continue;
                }
                uint64_t todo = __ballot(true);
                while(todo)
                {
                    const int leader = __builtin_ctzll(todo);
                    const uint32_t dl = (uint32_t)__builtin_amdgcn_readlane((int)d, leader);
                    const bool mine = d == dl;
                    const uint32_t sum = wave_sum_u32(mine ? cnt[u] : 0u);
                    if(lane == leader && sum)
                        atomicAdd(&hist[p * kBins32 + dl], sum);
                    todo &= ~__ballot(mine);
                }
            }
            const uint64_t occupied = __ballot(cnt[u] != 0);
            if(occupied && lane == 0)
                atomicMax(&s_last, t0 + u * kCoverThreads + wave * DSX_WAVE + 63 - __builtin_clzll(occupied));
            incl[u] = wave_incl_scan32(cnt[u], lane);
            if(lane == 63)
                wave_tot[u][wave] = incl[u];
        }
        __syncthreads();
#pragma unroll
        for(int u = 0; u < kTileRounds; ++u)
        {
            const int t = t0 + u * kCoverThreads + tid;
            if(t0 + u * kCoverThreads >= tiles)
                break;
            if(t < tiles)
                ranges[t] = (int32_t)(carry + sum_of_waves_before<kCoverThreads / DSX_WAVE>(wave_tot[u], wave) + incl[u] - cnt[u]);
            carry += sum_of_waves_before<kCoverThreads / DSX_WAVE>(wave_tot[u], kCoverThreads / DSX_WAVE);
        }
        __syncthreads();
    }
    __threadfence_block();
    __syncthreads();
    const int last = s_last;
    if(!J.plain)
    {
        const int32_t tail = last >= 0 ? ranges[last] : 0;
        for(int t = tid; t < tiles; t += kCoverThreads)
            if(t > last)
                ranges[t] = tail;
    }
    if(tid == 0)
    {
        ranges[tiles] = (int32_t)carry; // K
        if(J.last)
            *J.last = last;
        if(J.header)
            *J.header = J.header_value;
        for(int p = 0; p < plan.passes; ++p)
            atomicAdd(&hist[p * kBins32], negatives);
        if(wide_hist)
            wide_hist[0] = negatives;
    }
    __syncthreads();
    if(slot_hist)
        for(int j = tid; j < kMaxPasses32 * kBins32; j += kCoverThreads)
            slot_hist[j] = hist[j];
}

__global__ __launch_bounds__(kCoverThreads) void tile_counts_kernel(const CountsJobs jobs, int use_lds)
{
    extern __shared__ int32_t s_cells[];
    const CountsJob& J = jobs.job[blockIdx.x];
    int32_t* c = J.grid;
    if(use_lds)
    {
        const int cells = (J.ntx + 1) * (J.nty + 1) + 1;
        for(int j = threadIdx.x; j < cells; j += kCoverThreads)
            s_cells[j] = J.grid[j];
        c = s_cells;
        __syncthreads();
    }
    tile_counts(J, c);
}

// ---------------------------------------------------------------------------------------
// up to 131072 Gaussians: depth order, block offsets and counting in one launch
// ---------------------------------------------------------------------------------------
// Few keys are sorted by launches that wait for each other and do a microsecond's work each.  Here every workgroup finds out by
// itself which ranks are its own: it counts ALL keys into 4096 bins of their range (they lie in the L2), sums the bins up, and
// the keys between the bin borders next to ranks 512 w and 512 (w + 1) are workgroup w's, some 512 of them.  It reads the keys
// again, takes those, sorts them in LDS (2048 bins of its own part of the range, and a comparison with the few others in the
// same bin), and writes them where they belong: nobody waits for anybody.  Workgroups beside them fill corner grids and
// count the tiles and the bins.
// What is ordered are the distances of the depth keys from the smallest one with the Gaussian's index behind (all different).  Where a
// border would be kShareSlack or more ranks off (many equal or nearly equal depths) the bin before it is taken apart by the next
// twelve bits, if need be down to the index, so a workgroup never has more than 1023 keys, whatever they are.
// Bound by the two passes over all keys, of every workgroup, at some 35 bytes a cycle and compute unit, and by the chain around them:
// 2 K Gaussians 10 us (1 for the ranges, 1.5 for the two passes, 3 for borders and barriers, 2.5 in the sort, 2 until the last one has
// summed up), 16 K 11, 50 K 17.5, 100 K 23.5.  Before, a sort of 2048 keys in LDS and a merge up to 24576 Gaussians, the digit passes
// beyond: a whole forward of 16 K 78 -> 60 us, a training step of 50 K 199 -> 165, of 100 K 229 -> 198, 2 K 40 as it was.
constexpr int kRanksThreads = 1024;
static_assert(kRanksThreads == kCoverThreads && kRanksThreads == kHist32Threads, "tile_counts and load_keys are written for this many threads");
constexpr int kRanksBinBits = 12;
constexpr int kRanksBins = 1 << kRanksBinBits;
constexpr int kShareWanted = 512; // keys of a workgroup
constexpr int kShareSlack = 512;  // by so many fewer than this may its share begin and end late
constexpr int kShareMost = 1024;
constexpr int kShareBinBits = 11;
constexpr int kRanksWaves = kRanksThreads / DSX_WAVE;
// Rectangles that a grid's one workgroup counts alone: a thousand take it 0.4 us, and several workgroups pay for a grid in memory by its
// cells.  us of a whole forward, one workgroup -> eight: 640x480 5 K Gaussians 41.2 -> 42.4, 8 K 43.1 -> 42.8; 1280x720 5 K 49.0 -> 49.9,
// 12 K 53.7 -> 51.9; 1920x1080 8 K 52.4 -> 53.0, 12 K 55.5 -> 54.8; 2700x2300 12 K 101.2 -> 103.2, 24 K 112.4 -> 110.2; 3840x2160 3 K
// 100.1 -> 106.9, 18 K 122.7 -> 124.2, 24 K 129.5 -> 128.3.
constexpr int kCountAlone = 5500; // and one more for two cells
constexpr int kCountShare = 2048; // of each of several, at least
constexpr int kCountWorkgroupsMost = 32;
constexpr int kCellsAtOnce = 8; // cells of a grid in memory that a thread has on their way (one after the other: 12 K at 3840x2160 134 us, so 121)
static_assert(kShareWanted + kShareSlack <= kShareMost && kShareMost <= kRanksThreads, "a thread for each key");
static_assert(kShareWanted == 2 * kProjBlock && kRanksBins == 4 * kRanksThreads, "what the threads take");
constexpr size_t kRanksLds = (kRanksBins + DSX_WAVE) * 4 + 2 * kShareMost * 8;

struct RanksJob
{
    const uint32_t* depth_keys; // by Gaussian
    const uint2* rects;
    const uint2* key_ranges; // of 256 consecutive Gaussians (see OrderLayout)
    uint32_t* order;         // by depth
    uint2* rects_sorted;
    uint32_t* run_sums;   // pairs of 256 consecutive Gaussians in depth order (zero at first)
    uint32_t* block_sums; // their exclusive sums, and the total
    unsigned long long* key_count; // pairs of the tiles, of the bins; workgroups done: the order's, the tiles', the bins' (zero at first)
    int n, id_bits, shift, shares, counting; // counting: workgroups for each of the grids
    CountsJobs counts;
    HostCounts to_host;
};

// (the bits of a 64-bit number)
__device__ __forceinline__ int bits_of(uint64_t v)
{
    return v ? 64 - __builtin_clzll(v) : 0;
}

__device__ __forceinline__ void order_share(const RanksJob& J, const int share, uint32_t* const s_mem)
{
    uint32_t* const s_hist = s_mem;
    uint2* const s_rects = reinterpret_cast<uint2*>(s_mem + kRanksBins + DSX_WAVE);
    uint32_t* const s_taken_ids = reinterpret_cast<uint32_t*>(s_rects); // (before)
    uint64_t* const s_binned = reinterpret_cast<uint64_t*>(s_rects + kShareMost);
    __shared__ uint4 s_range[kRanksWaves];
    __shared__ __attribute__((aligned(16))) uint32_t s_tot[kRanksWaves];
    __shared__ uint32_t s_found[2][3], s_sums[kShareMost / kProjBlock + 2], s_taken;
    __shared__ unsigned long long s_all[kRanksWaves];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = J.n, blocks = (n + kProjBlock - 1) / kProjBlock;

    const KeyBatch ahead = load_keys(J.depth_keys, 0, n); // (the first ones, for every pass over the keys)
    // the keys' range, how many there are, and how many of the Gaussians before this workgroup's 512 emit
    uint32_t near16 = 0, far16 = 0, emit = 0, emit_before = 0;
    for(int b = tid; b < blocks; b += kRanksThreads)
    {
        const uint2 r = J.key_ranges[b];
        near16 = max(near16, r.x & 0xffffu);
        far16 = max(far16, r.y);
        emit += r.x >> 16;
        emit_before += b < 2 * share ? r.x >> 16 : 0u;
    }
    near16 = wave_incl_max_scan(near16);
    far16 = wave_incl_max_scan(far16);
    emit = wave_incl_scan_u32(emit);
    emit_before = wave_incl_scan_u32(emit_before);
    if(lane == 63)
        s_range[wave] = make_uint4(near16, far16, emit, emit_before);
    *reinterpret_cast<uint4*>(s_hist + 4 * tid) = make_uint4(0u, 0u, 0u, 0u);
    if(tid < kShareMost / kProjBlock + 2)
        s_sums[tid] = 0;
    if(tid == 0)
        s_taken = 0;
    __syncthreads();
    near16 = far16 = emit = emit_before = 0;
#pragma unroll
    for(int w = 0; w < kRanksWaves; ++w)
    {
        const uint4 r = s_range[w];
        near16 = max(near16, r.x);
        far16 = max(far16, r.y);
        emit += r.z;
        emit_before += r.w;
    }
    const uint32_t emitting = __builtin_amdgcn_readfirstlane(emit), before_mine = __builtin_amdgcn_readfirstlane(emit_before);
    const uint32_t lowest = 0xffffu - __builtin_amdgcn_readfirstlane(near16), highest = __builtin_amdgcn_readfirstlane(far16);
    const uint32_t first = emitting ? lowest << 16 : 0u;
    const int dist_bits = bits_of(emitting ? ((uint64_t)(highest - lowest + 1u) << 16) - 1u : 0xffffull); // (at least 16)
    const int id_bits = J.id_bits;
    // the number that is ordered: the distance, then the index
    auto number_of = [&](uint32_t key, int i) { return ((uint64_t)(key - first) << id_bits) | (uint32_t)i; };
    // a key that emits nothing has a distance like others only where the range ends at the largest number
    const bool apart = (uint64_t)first + (1ull << dist_bits) <= kNoPairsKey;
    // f(sixteen keys, the index of each) for all keys, those that emit nothing among them
    auto for_all = [&](auto f) {
        KeyBatch batch = ahead;
        for(int i0 = 0; i0 < n; i0 += kBatchKeys)
        {
            const KeyBatch next = load_keys(J.depth_keys, i0 + kBatchKeys, n);
#pragma unroll
            for(int b = 0; b < kBatchLoads; b += 4)
            {
                uint32_t key[16];
#pragma unroll
                for(int u = 0; u < 16; ++u)
                    key[u] = reinterpret_cast<const uint32_t*>(&batch.k[b + u / 4])[u % 4];
                f(key, [&](int u) { return i0 + 4 * ((b + u / 4) * kRanksThreads + tid) + u % 4; });
            }
            batch = next;
        }
    };
    // Behind a histogram of whole bins, `before` keys of which lie in front of it: for each rank of two, the first bin border at or
    // behind it (its number, its rank, and the rank of the border before it)
    auto borders = [&](uint32_t before, const uint32_t (&rank)[2]) {
        __syncthreads();
        const uint4 c = *reinterpret_cast<const uint4*>(s_hist + 4 * tid);
        const uint32_t count[4] = {c.x, c.y, c.z, c.w};
        const uint32_t sum = c.x + c.y + c.z + c.w, incl = wave_incl_scan_u32(sum);
        if(lane == 63)
            s_tot[wave] = incl;
        if(tid < 6)
            (&s_found[0][0])[tid] = tid % 3 ? before : 0u; // (rank 0: the first border)
        __syncthreads();
        uint32_t at = before + sum_of_waves_before<kRanksWaves>(s_tot, wave) + incl - sum;
#pragma unroll
        for(int u = 0; u < 4; ++u)
        {
#pragma unroll
            for(int e = 0; e < 2; ++e)
                if(at < rank[e] && rank[e] <= at + count[u])
                {
                    s_found[e][0] = 4 * tid + u + 1;
                    s_found[e][1] = at + count[u];
                    s_found[e][2] = at;
                }
            at += count[u];
        }
        __syncthreads();
    };

    const uint32_t rank[2] = {min((uint32_t)(kShareWanted * share), emitting), min((uint32_t)(kShareWanted * (share + 1)), emitting)};
    uint64_t border[2] = {0, 0};
    uint32_t place[2] = {0, 0};
    if(rank[0] < rank[1]) // (uniform; the last workgroups may have none)
    {
        // (keys that emit nothing are counted behind the bins, each lane's by themselves)
        const int top = dist_bits - kRanksBinBits;
        if(apart)
            for_all([&](const uint32_t (&key)[16], auto) {
#pragma unroll
                for(int u = 0; u < 16; ++u)
                    atomicAdd(&s_hist[min((key[u] - first) >> top, (uint32_t)(kRanksBins + lane))], 1u);
            });
        else
            for_all([&](const uint32_t (&key)[16], auto) {
#pragma unroll
                for(int u = 0; u < 16; ++u)
                    atomicAdd(&s_hist[key[u] == kNoPairsKey ? (uint32_t)(kRanksBins + lane) : (key[u] - first) >> top], 1u);
            });
        borders(0u, rank);
        uint32_t found[2][3];
#pragma unroll
        for(int e = 0; e < 6; ++e)
            found[e / 3][e % 3] = __builtin_amdgcn_readfirstlane((&s_found[0][0])[e]);
#pragma unroll
        for(int e = 0; e < 2; ++e)
        {
            int shift = dist_bits + id_bits - kRanksBinBits; // of the bins' numbers
            uint64_t low = 0;
            while(found[e][1] - rank[e] >= (uint32_t)kShareSlack && shift > 0)
            {
                // the bin in front of the border is a large one: bins of its own
                const int wide = shift;
                low += (uint64_t)(found[e][0] - 1u) << wide;
                shift = max(wide - kRanksBinBits, 0);
                __syncthreads();
                *reinterpret_cast<uint4*>(s_hist + 4 * tid) = make_uint4(0u, 0u, 0u, 0u);
                __syncthreads();
                for_all([&](const uint32_t (&key)[16], auto index) {
#pragma unroll
                    for(int u = 0; u < 16; ++u)
                    {
                        const uint64_t d = number_of(key[u], index(u)) - low;
                        if(key[u] != kNoPairsKey && (d >> wide) == 0)
                            atomicAdd(&s_hist[(uint32_t)(d >> shift)], 1u);
                    }
                });
                borders(found[e][2], rank);
#pragma unroll
                for(int j = 0; j < 3; ++j)
                    found[e][j] = __builtin_amdgcn_readfirstlane(s_found[e][j]);
            }
            border[e] = low + ((uint64_t)found[e][0] << shift);
            place[e] = found[e][1];
        }
        __syncthreads();

        // this workgroup's keys, in any order, and bins of their range
        // (a lane marks its sixteen keys and then stores the places of the few that are taken; one request for room a wavefront)
        auto take_all = [&](auto inside) {
            for_all([&](const uint32_t (&key)[16], auto index) {
                uint32_t marks = 0;
#pragma unroll
                for(int u = 0; u < 16; ++u)
                    marks += marks + (inside(key[u], index(u)) ? 1u : 0u);
                if(__builtin_amdgcn_ballot_w64(marks != 0) == 0)
                    return;
                const uint32_t taken = (uint32_t)__popc(marks), incl = wave_incl_scan_u32(taken);
                uint32_t at = 0;
                if(lane == 63)
                    at = atomicAdd(&s_taken, incl);
                at = (uint32_t)__builtin_amdgcn_readlane((int)at, 63) + incl - taken;
                while(marks != 0)
                {
                    const int u = 15 - (31 - __builtin_clz(marks));
                    marks ^= 0x8000u >> u;
                    s_taken_ids[min(at++, (uint32_t)kShareMost - 1u)] = (uint32_t)index(u);
                }
            });
        };
        const uint64_t ids = (1ull << id_bits) - 1;
        if(apart && ((border[0] | border[1]) & ids) == 0) // (the distances alone tell)
        {
            const uint32_t nearest = first + (uint32_t)(border[0] >> id_bits), depth = (uint32_t)((border[1] - border[0]) >> id_bits);
            take_all([&](uint32_t key, int) { return key - nearest < depth; });
        }
        else
            take_all([&](uint32_t key, int i) {
                const uint64_t number = number_of(key, i);
                return key != kNoPairsKey && number >= border[0] && number < border[1];
            });
        s_hist[tid] = s_hist[kRanksThreads + tid] = 0;
        __syncthreads();
        const int count = (int)(place[1] - place[0]);
        const int shift = max(bits_of(border[1] - border[0] - 1u) - kShareBinBits, 0);
        uint64_t mine = 0;
        uint32_t bin = 0, nth = 0;
        uint2 rect = make_uint2(0u, 0u);
        if(tid < count)
        {
            const int i = (int)s_taken_ids[tid];
            rect = J.rects[i]; // (here on time for the end)
            mine = number_of(J.depth_keys[i], i);
            bin = (uint32_t)((mine - border[0]) >> shift);
            nth = atomicAdd(&s_hist[bin], 1u);
        }
        __syncthreads();
        const uint2 c = *reinterpret_cast<const uint2*>(s_hist + 2 * tid);
        const uint32_t incl = wave_incl_scan_u32(c.x + c.y);
        if(lane == 63)
            s_tot[wave] = incl;
        __syncthreads();
        const uint32_t at = sum_of_waves_before<kRanksWaves>(s_tot, wave) + incl - c.x - c.y;
        *reinterpret_cast<uint2*>(s_hist + 2 * tid) = make_uint2(at, at + c.x);
        if(tid == 0)
            s_hist[1 << kShareBinBits] = (uint32_t)count;
        __syncthreads();
        uint32_t start = 0, end = 0;
        if(tid < count)
        {
            start = s_hist[bin];
            end = s_hist[bin + 1];
            s_binned[start + nth] = mine;
        }
        __syncthreads();
        uint32_t* const s_ids = s_hist;
        if(tid < count)
        {
            uint32_t r = start;
            for(uint32_t j = start; j < end; ++j)
                r += s_binned[j] < mine ? 1u : 0u;
            s_ids[r] = (uint32_t)mine & ((1u << id_bits) - 1u);
            s_rects[r] = rect;
        }
        __syncthreads();
        // the order, the rectangles in it, and the runs' sums
        const uint32_t p = place[0] + (uint32_t)tid, run0 = place[0] / kProjBlock;
        uint32_t pairs = 0;
        if(tid < count)
        {
            const uint2 r = s_rects[tid];
            J.order[p] = s_ids[tid];
            J.rects_sorted[p] = r;
            pairs = list_count(r, J.shift);
        }
        const uint32_t run = p / kProjBlock - run0, other = (uint32_t)__builtin_amdgcn_readlane((int)run, 63);
        if(__builtin_amdgcn_readfirstlane(run) == other)
        {
            const uint32_t sum = wave_sum_u32(pairs);
            if(lane == 0 && sum)
                atomicAdd(&s_sums[run], sum);
        }
        else if(pairs)
            atomicAdd(&s_sums[run], pairs);
        __syncthreads();
        uint32_t done = 0;
        if(tid < kShareMost / kProjBlock + 2 && s_sums[tid])
            done = atomicAdd(&J.run_sums[run0 + tid], s_sums[tid]);
        asm volatile("s_waitcnt vmcnt(0)" ::"v"(done) : "memory"); // (an addition has been performed when its result is back)
    }
    // of the Gaussians 512 w to 512 w + 511 those that emit nothing: behind the others, by index
    {
        const int i = kShareWanted * share + tid;
        const bool none = tid < kShareWanted && i < n && J.depth_keys[min(i, n - 1)] == kNoPairsKey;
        const uint64_t m = __builtin_amdgcn_ballot_w64(none);
        __syncthreads();
        if(lane == 0)
            s_tot[wave] = (uint32_t)__popcll(m);
        __syncthreads();
        if(none)
        {
            const uint32_t at = emitting + (uint32_t)(kShareWanted * share) - before_mine +
                                sum_of_waves_before<kRanksWaves>(s_tot, wave) + bits_below(m);
            J.order[at] = (uint32_t)i;
            J.rects_sorted[at] = make_uint2(0u, 0u);
        }
    }
    // the last workgroup turns the runs' sums into the places where they begin
    if(tid == 0)
        s_last = atomicAdd(J.key_count + 2, 1ull) == (unsigned long long)(J.shares - 1);
    __syncthreads();
    if(!s_last)
        return;
    static_assert(kRanksMax / kProjBlock <= kRanksThreads, "a thread for each run");
    const uint32_t sum = tid < blocks ? atomicAdd(&J.run_sums[tid], 0u) : 0u;
    const uint32_t incl = wave_incl_scan_u32(sum);
    unsigned long long all = sum; // (64 bits: what does not fit 32 is refused by the callers, but must not look like less)
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        all += __shfl_xor(all, o, DSX_WAVE);
    if(lane == 63)
    {
        s_tot[wave] = incl;
        s_all[wave] = all;
    }
    __syncthreads();
    if(tid < blocks)
        J.block_sums[tid] = sum_of_waves_before<kRanksWaves>(s_tot, wave) + incl - sum;
    if(tid == 0)
    {
        all = 0;
        for(int w = 0; w < kRanksWaves; ++w)
            all += s_all[w];
        J.block_sums[blocks] = all > 0xffffffffull ? 0xffffffffu : (uint32_t)all;
    }
}

// the corner grid of the rectangles (of their bins when `bins`) in LDS, one of `parts` shares of them; then, by the workgroup
// that is last to add its own to the whole grid: the pairs' number to the host, the counts
__device__ __forceinline__ void count_share(const RanksJob& J, const bool bins, const int part, const int parts, int32_t* s_grid)
{
    __shared__ unsigned long long s_pairs;
    __shared__ int s_is_last;
    const CountsJob& C = J.counts.job[bins ? 1 : 0];
    const int tid = threadIdx.x;
    const int pitch = C.ntx + 1, cells = pitch * (C.nty + 1) + 1;
    for(int j = tid; j < (cells + 3) / 4; j += kRanksThreads)
        reinterpret_cast<int4*>(s_grid)[j] = make_int4(0, 0, 0, 0);
    if(tid == 0)
        s_pairs = 0ull;
    __syncthreads();
    unsigned long long pairs = 0;
    for(int g = part * kRanksThreads + tid; g < J.n; g += parts * kRanksThreads)
    {
        const uint2 r = J.rects[g];
        int w = (int)(r.y & 0xffffu), h = (int)((r.y >> 16) & 0x7fffu);
        if(w == 0 || h == 0)
            continue;
        int sx = (int)(r.x & 0xffffu), sy = (int)(r.x >> 16);
        if(r.y >> 31)
        {
            pairs += (unsigned long long)(w * h);
            atomicAdd(&s_grid[cells - 1], w * h);
            continue;
        }
        if(bins)
        {
            const BinRect b = bin_rect(r, J.shift);
            sx = (int)b.bx;
            sy = (int)b.by;
            w = (int)b.bw;
            h = (int)b.bh;
        }
        pairs += (unsigned long long)(w * h);
        atomicAdd(&s_grid[sy * pitch + sx], 1);
        atomicAdd(&s_grid[sy * pitch + sx + w], -1);
        atomicAdd(&s_grid[(sy + h) * pitch + sx], -1);
        atomicAdd(&s_grid[(sy + h) * pitch + sx + w], 1);
    }
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        pairs += __shfl_xor(pairs, o, DSX_WAVE);
    if((tid & 63) == 0 && pairs)
        atomicAdd(&s_pairs, pairs);
    __syncthreads();
    if(parts > 1)
    {
        // (an addition has been performed when its result is back; every wavefront's are before the barrier)
        int32_t back = 0;
        for(int j0 = tid; j0 < cells; j0 += kCellsAtOnce * kRanksThreads)
        {
            int32_t mine[kCellsAtOnce], was[kCellsAtOnce];
#pragma unroll
            for(int u = 0; u < kCellsAtOnce; ++u)
                mine[u] = j0 + u * kRanksThreads < cells ? s_grid[j0 + u * kRanksThreads] : 0;
#pragma unroll
            for(int u = 0; u < kCellsAtOnce; ++u)
            {
                was[u] = 0;
                if(mine[u])
                    was[u] = atomicAdd(&C.grid[j0 + u * kRanksThreads], mine[u]);
            }
#pragma unroll
            for(int u = 0; u < kCellsAtOnce; ++u)
                back |= was[u];
        }
        unsigned long long pairs_back = 0;
        if(tid == 0)
            pairs_back = atomicAdd(J.key_count + (bins ? 1 : 0), s_pairs);
        asm volatile("s_waitcnt vmcnt(0)" ::"v"(back), "v"(pairs_back) : "memory");
        __syncthreads();
        if(tid == 0)
        {
            s_is_last = atomicAdd(J.key_count + (bins ? 4 : 3), 1ull) == (unsigned long long)(parts - 1);
            if(s_is_last)
                s_pairs = atomicAdd(J.key_count + (bins ? 1 : 0), 0ull);
        }
        __syncthreads();
        if(!s_is_last)
            return;
        for(int j0 = tid; j0 < cells; j0 += kCellsAtOnce * kRanksThreads)
        {
            int32_t sum[kCellsAtOnce];
#pragma unroll
            for(int u = 0; u < kCellsAtOnce; ++u)
                sum[u] = __hip_atomic_load(C.grid + min(j0 + u * kRanksThreads, cells - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for(int u = 0; u < kCellsAtOnce; ++u)
                if(j0 + u * kRanksThreads < cells)
                    s_grid[j0 + u * kRanksThreads] = sum[u];
        }
        __syncthreads();
    }
    if(tid == 0 && J.to_host.words)
    {
        store_to_host(J.to_host, bins ? 1 : 0, s_pairs);
        if(J.shift == 0)
            store_to_host(J.to_host, 1, 0ull);
    }
    tile_counts(C, s_grid);
}

__global__ __launch_bounds__(kRanksThreads) void order_ranks_kernel(const RanksJob J)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t s_ranks[];
    // (the counting first: the host waits for its sums)
    const int counting = J.counting * (J.shift ? 2 : 1), w = (int)blockIdx.x;
    if(w < counting)
        count_share(J, w >= J.counting, w % J.counting, J.counting, reinterpret_cast<int32_t*>(s_ranks));
    else
        order_share(J, w - counting, s_ranks);
}

// true: done (or failed: *rc).  false: too many Gaussians, or a corner grid that does not fit the LDS
static bool launch_order_ranks(const ListGrid& lg, int64_t n, char* base, const OrderLayout& o, const HostCounts& to_host,
                               const CountsJobs& jobs, hipStream_t stream, int* rc)
{
    const int cells = (lg.ntx + 1) * (lg.nty + 1) + 1;
    if(n > kRanksMax || cells > kCoverLdsCellsLarge - 4096) // (less what the kernel has besides)
        return false;
    const size_t bytes = std::max(kRanksLds, ((size_t)cells * 4 + 15) & ~(size_t)15);
    if(bytes > 65536 - 8192 &&
       hipFuncSetAttribute(reinterpret_cast<const void*>(order_ranks_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)bytes) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    RanksJob J;
    J.depth_keys = reinterpret_cast<const uint32_t*>(base + o.depth_keys);
    J.rects = reinterpret_cast<const uint2*>(base + o.rects);
    J.key_ranges = reinterpret_cast<const uint2*>(base + o.key_ranges);
    J.order = reinterpret_cast<uint32_t*>(base + o.ids_a);
    J.rects_sorted = reinterpret_cast<uint2*>(base + o.rects_sorted);
    J.run_sums = reinterpret_cast<uint32_t*>(base + o.run_sums);
    J.block_sums = reinterpret_cast<uint32_t*>(base + o.block_sums);
    J.key_count = reinterpret_cast<unsigned long long*>(base + o.key_count);
    J.n = (int)n;
    J.id_bits = std::max(1, 64 - __builtin_clzll((unsigned long long)std::max<int64_t>(n - 1, 1)));
    J.shift = lg.shift;
    J.shares = (int)((n + kShareWanted - 1) / kShareWanted);
    J.counting = n <= kCountAlone + cells / 2 ? 1 : (int)std::min<int64_t>(kCountWorkgroupsMost, (n + kCountShare - 1) / kCountShare);
    J.counts = jobs;
    J.to_host = to_host;
    {
        DSX_TIMED("order_ranks_kernel", stream);
        hipLaunchKernelGGL(order_ranks_kernel, dim3(J.shares + J.counting * (lg.shift ? 2 : 1)), dim3(kRanksThreads), bytes, stream, J);
    }
    *rc = hipGetLastError() == hipSuccess ? DSX_OK : DSX_ERR_LAUNCH;
    return true;
}

// the counting of the tiles and, for binned lists, of the bins
static CountsJobs counts_jobs(const ListGrid& lg, int64_t n, char* base, const OrderLayout& o)
{
    const RangesLayout rl = ranges_layout(lg);
    int32_t* const ranges = reinterpret_cast<int32_t*>(base + o.ranges);
    CountsJobs jobs;
    CountsJob& fine = jobs.job[0];
    fine.grid = reinterpret_cast<int32_t*>(base + o.cover);
    fine.ntx = lg.ntx;
    fine.nty = lg.nty;
    fine.plain = 0;
    fine.plan = partition_digits(slot_bits(lg.tiles()), wide_digit_most(slot_bits(lg.tiles()), n, false) > 0);
    fine.slot_hist = lg.shift ? nullptr : reinterpret_cast<uint32_t*>(base + o.slot_hist);
    fine.ranges = ranges + rl.fine;
    fine.last = lg.shift ? ranges + rl.last_tile : nullptr;
    fine.header = ranges + rl.header;
    fine.header_value = lg.shift;
    jobs.job[1] = fine;
    if(lg.shift)
    {
        CountsJob& bins = jobs.job[1];
        bins.grid = reinterpret_cast<int32_t*>(base + o.bin_cover);
        bins.ntx = lg.nbx;
        bins.nty = lg.nby;
        bins.plain = 1;
        bins.plan = partition_digits(slot_bits(lg.bins()), wide_digit_most(slot_bits(lg.bins()), n, true) > 0);
        bins.slot_hist = reinterpret_cast<uint32_t*>(base + o.slot_hist);
        bins.ranges = ranges + rl.bins;
        bins.last = nullptr;
        bins.header = nullptr;
    }
    return jobs;
}

// order: the buffer of order_layout(n) whose depth_keys and rects the projection has written
void depth_order_clear_region(const dsx_camera& cam, int64_t n, void* order, uint32_t** words, int64_t* count)
{
    // the sort's histograms, counters and look-back statuses and, right behind them, the corner grid
    const OrderLayout o = order_layout(n, cam.image_width, cam.image_height, camera_bin(cam));
    const Sort32Workspace w = sort32_workspace(n, 32, sort32_tile_keys(n));
    *words = reinterpret_cast<uint32_t*>(static_cast<char*>(order) + o.sort + w.hist);
    *count = (int64_t)((w.bytes + (o.ranges - o.cover)) / 4);
}

// The form of the scatter: as many Gaussians to a workgroup as leave one for each compute unit
struct ScatterForm
{
    void (*kernel)(BucketsJob);
    int bin_bits, tile; // Gaussians of a workgroup
    size_t bytes;       // of LDS
};
static ScatterForm scatter_form(int64_t n)
{
    auto form = [](void (*kernel)(BucketsJob), int runs, int bin_bits) {
        return ScatterForm{kernel, bin_bits, runs * kScatterWaves * kProjBlock, (size_t)kBucketsMost * 12 + ((size_t)2 << bin_bits)};
    };
    if(n <= 1 << 20)
        return form(depth_scatter_kernel<1, 12>, 1, 12);
    if(n <= 2 << 20)
        return form(depth_scatter_kernel<2, 13>, 2, 13);
    if(n <= 3 << 20)
        return form(depth_scatter_kernel<3, 13>, 3, 13);
    if(n <= 4 << 20)
        return form(depth_scatter_kernel<4, 13>, 4, 13);
    return form(depth_scatter_kernel<4, 14>, 4, 14);
}

// What the buckets' launches work on; returns the bits of the bins, or 0 where a kernel cannot have the LDS that it needs: the passes
// run then.
static int buckets_job(int64_t n, const ScatterForm& scatter, char* base, const OrderLayout& o, int shift, const HostCounts& to_host,
                       BucketsJob* J)
{
    const int bin_bits = scatter.bin_bits;
    // (a few hundred buckets at least)
    J->bucket_bits = n > 1 << 19 ? kBucketBitsMost : kBucketBitsMost - 1;
    J->buckets = (int)((n + (1 << J->bucket_bits) - 1) >> J->bucket_bits);
    J->n = (int)n;
    J->shift = shift;
    J->to_host = to_host;
    char* at = base + o.buckets;
    auto take = [&](size_t bytes) {
        char* const mine = at;
        at += (bytes + 255) & ~(size_t)255;
        return mine;
    };
    J->bins = reinterpret_cast<uint32_t*>(take((size_t)4 << kDepthBinBitsMost));
    J->cursors = reinterpret_cast<unsigned long long*>(take((size_t)kBucketsMost * 8));
    J->done = reinterpret_cast<uint32_t*>(take(8));
    J->starts = reinterpret_cast<uint2*>(take((size_t)(kBucketsMost + 1) * 8));
    J->span = reinterpret_cast<uint32_t*>(take((kSpanWords + kSpanChunks) * 4));
    J->digits = reinterpret_cast<uint32_t*>(base + o.sort + sort32_workspace(n, 32, sort32_tile_keys(n)).hist);
    J->keys = reinterpret_cast<const uint32_t*>(base + o.depth_keys);
    J->rects = reinterpret_cast<const uint2*>(base + o.rects);
    J->key_ranges = reinterpret_cast<const uint2*>(base + o.key_ranges);
    J->records = reinterpret_cast<Words4*>(base + o.records);
    J->order = reinterpret_cast<uint32_t*>(base + o.ids_a);
    J->rects_sorted = reinterpret_cast<uint2*>(base + o.rects_sorted);
    J->block_sums = reinterpret_cast<uint32_t*>(base + o.block_sums);
    auto allow = [](const void* kernel, size_t bytes, size_t own) {
        return bytes + own <= 65536 || hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
    };
    if(!allow(reinterpret_cast<const void*>(depth_hist_kernel), (size_t)4 << bin_bits, 1024) ||
       !allow(reinterpret_cast<const void*>(scatter.kernel), scatter.bytes, 1024))
    {
        (void)hipGetLastError();
        *J = {};
        return 0;
    }
    return bin_bits;
}

// Is the second launch of the buckets made before the host knows whether there are any?  The first one tells it a few us after it began:
// where it is short the second would come late (without: 140 K 112 -> 119 us a forward, 300 K 149 -> 153, 1 M 247 -> 249, 3 M 360 ->
// 360); where there are none an empty launch takes 4 us, and a wide range is what crowds the bins.
static bool launches_both(int64_t n, const DepthRange& range)
{
    return n <= 1 << 19 || (n <= 1 << 20 && range.behind < 6u << 23);
}

// The depth sort of a whole forward (cleared workspace): its first launch, which tells the host the range,
struct DepthSort
{
    BucketsJob buckets = {};
    ScatterForm scatter = {};
    int bin_bits = 0; // 0: no buckets
};
static int launch_depth_hist(int64_t n, char* base, const OrderLayout& o, int64_t blocks, bool by_buckets, int list_shift,
                             const HostCounts& to_host, hipStream_t stream, DepthSort* sort)
{
    if(n >= (1ll << 30))
        return DSX_ERR_TOO_LARGE;
    const int64_t chunks = (n + kHist32Threads * kDepthHistItems - 1) / (kHist32Threads * kDepthHistItems);
    sort->scatter = scatter_form(n);
    sort->bin_bits = by_buckets ? buckets_job(n, sort->scatter, base, o, list_shift, to_host, &sort->buckets) : 0;
    const size_t bytes = std::max(kSortWordsMost, sort->bin_bits ? (size_t)1 << sort->bin_bits : 0) * 4;
    DSX_TIMED("depth_hist_kernel", stream);
    hipLaunchKernelGGL(depth_hist_kernel, dim3((unsigned)min((int64_t)DSX_HIST_BLOCKS, chunks)), dim3(kHist32Threads), bytes, stream,
                       reinterpret_cast<const uint32_t*>(base + o.depth_keys), n, reinterpret_cast<const uint2*>(base + o.key_ranges), blocks,
                       reinterpret_cast<uint32_t*>(base + o.sort + sort32_workspace(n, 32, sort32_tile_keys(n)).hist), sort->buckets.bins,
                       sort->bin_bits, sort->buckets.span, to_host);
    DSX_LAUNCH_CHECK();
    return DSX_OK;
}

// and the others: ids in `ids_a`, the rectangles of the first `emitting` of them in `rects_sorted`.
static int launch_depth_sort(int64_t n, char* base, const OrderLayout& o, bool carry, const DepthSort& sort, const HostCounts& to_host,
                             int polls, hipStream_t stream, int64_t* emitting, bool* offsets_done)
{
    uint32_t* const keys_a = reinterpret_cast<uint32_t*>(base + o.depth_keys);
    uint32_t* const keys_b = reinterpret_cast<uint32_t*>(base + o.keys_alt);
    uint32_t* const ids_a = reinterpret_cast<uint32_t*>(base + o.ids_a);
    uint32_t* const ids_b = reinterpret_cast<uint32_t*>(base + o.ids_b);
    const uint2* const rects = reinterpret_cast<const uint2*>(base + o.rects);
    uint2* const rects_sorted = reinterpret_cast<uint2*>(base + o.rects_sorted);
    uint32_t* const packed_a = reinterpret_cast<uint32_t*>(base + o.rects_sorted);
    uint32_t* const packed_b = reinterpret_cast<uint32_t*>(base + o.rects32);
    char* const ws = base + o.sort;
    const Sort32Workspace w = sort32_workspace(n, 32, sort32_tile_keys(n));
    const BucketsJob& buckets = sort.buckets;
    const ScatterForm& scatter = sort.scatter;
    uint64_t ends, emitters;
    if(!wait_for_word(to_host, 2, stream, &ends) || !wait_for_word(to_host, 3, stream, &emitters))
        return DSX_ERR_RUNTIME;
    const DepthRange range = depth_range((uint32_t)(ends & 0xffffu), (uint32_t)(ends >> 16));
    if(sort.bin_bits && depth_bins(range))
    {
        {
            DSX_TIMED("depth_scatter_kernel", stream);
            hipLaunchKernelGGL(scatter.kernel, dim3((unsigned)((n + scatter.tile - 1) / scatter.tile)), dim3(kScatterThreads), scatter.bytes,
                               stream, buckets);
        }
        DSX_LAUNCH_CHECK();
        auto sort_buckets = [&]() {
            if(emitters == 0)
                return;
            DSX_TIMED("order_buckets_kernel", stream);
            hipLaunchKernelGGL(order_buckets_kernel, dim3((unsigned)((emitters + (1ull << buckets.bucket_bits) - 1) >> buckets.bucket_bits)),
                               dim3(kBucketThreads), 0, stream, buckets);
        };
        const bool at_once = launches_both(n, range);
        if(at_once)
            sort_buckets();
        uint64_t answer;
        if(!wait_for_word(to_host, 4, stream, &answer))
            return DSX_ERR_RUNTIME;
        if(answer == kBucketsDone)
        {
            *offsets_done = true;
            if(!at_once)
                sort_buckets();
            DSX_LAUNCH_CHECK();
            return DSX_OK;
        }
        // too many keys in a bin: the passes, whose digits have been counted
    }
    const char* const label = "onesweep32_kernel<sort>";
    *emitting = (int64_t)emitters;
    if(!range.narrow)
    {
        // (four passes: the values, iota in the first, go b, a, b, a and end in ids_a)
        uint32_t *ko, *vo;
#define DSX_DEPTH_SORT_ITEMS(ITEMS)                                                                                     \
    case ITEMS:                                                                                                        \
        return carry ? sort32_passes<uint32_t, kSortThreads32, ITEMS, true>(n, 32, keys_a, ids_a, keys_b, ids_b, true,  \
                                                                            false, ws, label, stream, &ko, &vo, rects, \
                                                                            rects_sorted, nullptr, packed_a, packed_b, \
                                                                            polls)                                     \
                     : sort32_passes<uint32_t, kSortThreads32, ITEMS>(n, 32, keys_a, ids_a, keys_b, ids_b, true, false, \
                                                                      ws, label, stream, &ko, &vo, rects, rects_sorted, \
                                                                      nullptr, nullptr, nullptr, polls)
        switch(sort32_items(n))
        {
            DSX_DEPTH_SORT_ITEMS(1);
            DSX_DEPTH_SORT_ITEMS(2);
            DSX_DEPTH_SORT_ITEMS(3);
            DSX_DEPTH_SORT_ITEMS(4);
            DSX_DEPTH_SORT_ITEMS(6);
            DSX_DEPTH_SORT_ITEMS(8);
            DSX_DEPTH_SORT_ITEMS(kSortItemsMax32);
        }
#undef DSX_DEPTH_SORT_ITEMS
        return DSX_ERR_RUNTIME;
    }
    // Three passes, of which the first puts the Gaussians that emit nothing into their final places (in ids_a, where its
    // values and the last pass's go) and the others sort the rest: a third fewer keys where a third of the cloud is out of sight.
    // The last pass never reads packed rectangles from the memory that it unpacks them into.
    *emitting = (int64_t)emitters;
    uint32_t* const counters = reinterpret_cast<uint32_t*>(ws + w.counters);
    int64_t count = n;
    int items = sort32_items(n);
    for(int p = 0; p < kDepthPasses; ++p)
    {
        const bool first = p == 0, last = p == kDepthPasses - 1;
        if(p == 1)
        {
            // (as few keys to a thread as the statuses of n Gaussians' tiles have room for)
            count = *emitting;
            const int family[] = {1, 2, 3, 4, 6, 8, kSortItemsMax32};
            for(int i : family)
                if((items = i) >= sort32_items(count) && (count + (int64_t)i * kSortThreads32 - 1) / ((int64_t)i * kSortThreads32) <= w.tiles)
                    break;
        }
        const unsigned tiles = (unsigned)((count + (int64_t)items * kSortThreads32 - 1) / ((int64_t)items * kSortThreads32));
        if(tiles == 0)
            break;
        RectJob job = {};
        if(carry)
        {
            job.pack_src = first ? rects : nullptr;
            job.carry_in = p & 1 ? packed_a : packed_b;
            job.carry_out = p & 1 ? packed_b : packed_a;
            job.unpack_dst = last ? rects_sorted : nullptr;
        }
        else if(last)
        {
            job.gather_src = rects;
            job.gather_dst = rects_sorted;
            job.last_value = (uint32_t)(n - 1);
        }
        const KeyRange keys = {range.first, range.behind, (uint32_t)*emitting};
        const uint32_t* const keys_in = p & 1 ? keys_b : keys_a;
        uint32_t* const keys_out = last ? nullptr : (p & 1 ? keys_a : keys_b);
        const uint32_t* const vals_in = first ? nullptr : (p & 1 ? ids_a : ids_b);
        uint32_t* const vals_out = p & 1 ? ids_b : ids_a;
        DSX_TIMED(label, stream);
        const uint32_t* const counts = reinterpret_cast<const uint32_t*>(ws + w.hist) + p * kDepthBins;
        uint32_t* const status = reinterpret_cast<uint32_t*>(ws + w.status) + (size_t)p * w.tiles * kDepthBins;
#define DSX_DEPTH_PASS(ITEMS, CARRY)                                                                                    \
    if(first)                                                                                                           \
        hipLaunchKernelGGL((onesweep32_first_kernel<ITEMS, CARRY>), dim3(tiles), dim3(kSortThreads32), 0, stream,        \
                           keys_in, keys_out, vals_out, count, range.digits.shift[p], range.digits.mask[p], counts,     \
                           status, counters + p, counters + w.passes, polls, job, keys);                                \
    else                                                                                                                \
        hipLaunchKernelGGL((onesweep32_kernel<uint32_t, kSortThreads32, ITEMS, CARRY, kDepthBits>), dim3(tiles),         \
                           dim3(kSortThreads32), 0, stream, keys_in, vals_in, keys_out, vals_out, count,                \
                           range.digits.shift[p], range.digits.mask[p], counts, status, counters + p,                  \
                           counters + w.passes, polls, job)
#define DSX_DEPTH_PASS_ITEMS(ITEMS)         \
    case ITEMS:                             \
        if(carry)                           \
        {                                   \
            DSX_DEPTH_PASS(ITEMS, true);    \
        }                                   \
        else                                \
        {                                   \
            DSX_DEPTH_PASS(ITEMS, false);   \
        }                                   \
        break
        switch(items)
        {
            DSX_DEPTH_PASS_ITEMS(1);
            DSX_DEPTH_PASS_ITEMS(2);
            DSX_DEPTH_PASS_ITEMS(3);
            DSX_DEPTH_PASS_ITEMS(4);
            DSX_DEPTH_PASS_ITEMS(6);
            DSX_DEPTH_PASS_ITEMS(8);
            DSX_DEPTH_PASS_ITEMS(kSortItemsMax32);
        }
#undef DSX_DEPTH_PASS_ITEMS
#undef DSX_DEPTH_PASS
        DSX_LAUNCH_CHECK();
    }
    return DSX_OK;
}

// to_host (optional): words of pinned host memory that receive the pair counts (per-tile lists: what the
// reference calls K, the fine ranges and final_idx index that many pairs; bin lists, zero when the lists
// are per tile) as soon as the rectangles have been counted, while the sort still runs.
int launch_depth_order(const dsx_camera& cam, int64_t n, void* order, hipStream_t stream, bool already_cleared,
                       HostCounts to_host, int sort_polls, int offset_polls)
{
    if(n <= 0)
        return DSX_OK;
    const OrderLayout o = order_layout(n, cam.image_width, cam.image_height, camera_bin(cam));
    char* base = static_cast<char*>(order);
    uint32_t* keys_a = reinterpret_cast<uint32_t*>(base + o.depth_keys);
    uint32_t* keys_b = reinterpret_cast<uint32_t*>(base + o.keys_alt);
    uint32_t* ids_a = reinterpret_cast<uint32_t*>(base + o.ids_a);
    uint32_t* ids_b = reinterpret_cast<uint32_t*>(base + o.ids_b);
    uint32_t* block_sums = reinterpret_cast<uint32_t*>(base + o.block_sums);
    // one fill zeroes the sort's counters and, right behind them, the corner grid
    int rc = DSX_OK;
    if(!already_cleared)
    {
        uint32_t* words;
        int64_t count;
        depth_order_clear_region(cam, n, order, &words, &count);
        rc = launch_fill_u32(words, count, 0u, stream);
    }
    if(rc)
        return rc;

    const CountsJobs jobs = counts_jobs(list_grid(cam), n, base, o);
    // (limits of its waits: asked for are the kernels that wait)
    if(sort_polls == kSpinLimit32 && offset_polls == kSpinLimit32 &&
       launch_order_ranks(list_grid(cam), n, base, o, to_host, jobs, stream, &rc))
        return rc;

    // pairs per tile: digit histograms of the tile partition and the tile ranges that the second
    // half of the forward needs.  They depend on the rectangles only, not on the depth order,
    // so they run on the helper stream beside the sort (fork after the fill, join at the end).
    hipStream_t side = helper_stream();
    hipEvent_t fork = nullptr, join = nullptr;
    if(side && (hipEventCreateWithFlags(&fork, hipEventDisableTiming) != hipSuccess ||
                hipEventCreateWithFlags(&join, hipEventDisableTiming) != hipSuccess || hipEventRecord(fork, stream) != hipSuccess))
    {
        (void)hipGetLastError();
        side = nullptr;
    }
    // (a wait for the range: what few Gaussians need is done before the host could have launched the rest.  Beyond those of
    // launch_order_ranks it pays where buckets order them, a forward of 150 K 120 -> 100 us.  The launch that tells the host goes out
    // before those of the helper stream: us of a forward of 140 K to 260 K that is waited for 3 to 9 less.  Where the range has both
    // signs a forward of so many at 640x480 takes 138 to 141 among others and 164 to 162 alone, at 1280x720 168 to 168 and 193 to 188.)
    const int64_t blocks = (n + kProjBlock - 1) / kProjBlock;
    const bool by_buckets = orders_by_buckets(n) && sort_polls == kSpinLimit32 && offset_polls == kSpinLimit32;
    const bool by_range = to_host.words && (sort32_items(n) > 1 || by_buckets);
    DepthSort sort;
    if(by_range)
        rc = launch_depth_hist(n, base, o, blocks, by_buckets, list_grid(cam).shift, to_host, stream, &sort);
    if(side && hipStreamWaitEvent(side, fork, 0) != hipSuccess)
    {
        (void)hipGetLastError();
        side = nullptr;
    }
    {
        hipStream_t cs = side ? side : stream;
        const ListGrid lg = list_grid(cam);
        const int ntx = lg.ntx, nty = lg.nty;
        const int cells = (ntx + 1) * (nty + 1) + 1;
        const int bcells = lg.shift ? (lg.nbx + 1) * (lg.nby + 1) + 1 : 0;
        int32_t* grid = reinterpret_cast<int32_t*>(base + o.cover);
        int32_t* bin_grid = reinterpret_cast<int32_t*>(base + o.bin_cover);
        // The corner grids are privatised in LDS whenever they fit (a 4K image has 32 776 cells =
        // 128 KB: one workgroup per CU); beyond 64 KB a kernel needs its limit raised first.
        // Global atomics are the fallback: correct for any grid, but 24 M same-line atomics
        // at 6 M Gaussians cost 0.6 ms and stall the sort passes that run beside them.
        int use_lds = cells + bcells <= kCoverLdsCells ? 1 : 0;
        if(!use_lds && cells + bcells <= kCoverLdsCellsLarge)
        {
            const int bytes = (cells + bcells) * 4;
            use_lds = hipFuncSetAttribute(reinterpret_cast<const void*>(tile_cover_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess &&
                              hipFuncSetAttribute(reinterpret_cast<const void*>(tile_counts_kernel),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess
                          ? 1
                          : 0;
            if(!use_lds)
                (void)hipGetLastError();
        }
        const int64_t want = (n + kCoverThreads - 1) / kCoverThreads;
        {
            DSX_TIMED("tile_cover_kernel", cs);
            hipLaunchKernelGGL(tile_cover_kernel, dim3((unsigned)min((int64_t)kCoverBlocks, want)), dim3(kCoverThreads),
                               use_lds ? (size_t)(cells + bcells) * 4 : 0, cs,
                               reinterpret_cast<const uint2*>(base + o.rects), n, ntx, nty, lg.shift, lg.nbx, lg.nby,
                               use_lds, grid, bin_grid, reinterpret_cast<unsigned long long*>(base + o.key_count),
                               to_host);
        }
        {
            DSX_TIMED("tile_counts_kernel", cs);
            hipLaunchKernelGGL(tile_counts_kernel, dim3(lg.shift ? 2 : 1), dim3(kCoverThreads),
                               use_lds ? (size_t)cells * 4 : 0, cs, jobs, use_lds);
        }
    }
    bool joined = true;
    if(side)
        joined = hipEventRecord(join, side) == hipSuccess;
    // the caller's stream takes the helper's work back in before this function returns
    auto finish = [&](int status) {
        if(side && joined)
            joined = hipStreamWaitEvent(stream, join, 0) == hipSuccess;
        if(fork)
            (void)hipEventDestroy(fork);
        if(join)
            (void)hipEventDestroy(join);
        return status ? status : (joined ? DSX_OK : DSX_ERR_RUNTIME);
    };
    if(hipGetLastError() != hipSuccess)
        return finish(DSX_ERR_LAUNCH);

    uint32_t *ko, *vo = ids_a;
    int64_t emitting = n;
    // the rectangles travel through the passes when they pack into 32 bits (the passes end in
    // rects_sorted, whose first half holds the packed ones of the passes in between), else the last
    // pass gathers them
    const bool carry = tiles_x(cam.image_width) <= kRect32MaxTiles && tiles_y(cam.image_height) <= kRect32MaxTiles;
    bool offsets_done = false;
    if(rc)
        return finish(rc);
    if(by_range)
        rc = launch_depth_sort(n, base, o, carry, sort, to_host, sort_polls, stream, &emitting, &offsets_done);
    else // (four passes: the values, iota in the first, go b, a, b, a and end in ids_a)
        rc = launch_sort32(n, 32, keys_a, ids_a, keys_b, ids_b, true, false, base + o.sort, stream, &ko, &vo,
                       reinterpret_cast<const uint2*>(base + o.rects), reinterpret_cast<uint2*>(base + o.rects_sorted),
                       true, carry ? reinterpret_cast<uint32_t*>(base + o.rects_sorted) : nullptr,
                       carry ? reinterpret_cast<uint32_t*>(base + o.rects32) : nullptr, sort_polls);
    if(rc)
        return finish(rc);
    if(vo != ids_a)
        return finish(DSX_ERR_RUNTIME);
    if(!offsets_done)
    {
        DSX_TIMED("ordered_offsets_kernel", stream);
        hipLaunchKernelGGL(ordered_offsets_kernel, dim3((unsigned)((n + kOffsetsShare - 1) / kOffsetsShare)), dim3(kOffsetsThreads), 0, stream,
                           reinterpret_cast<uint2*>(base + o.rects_sorted), n, emitting, list_grid(cam).shift, block_sums,
                           reinterpret_cast<unsigned long long*>(base + o.offsets), offset_polls);
    }
    return finish(hipGetLastError() != hipSuccess ? DSX_ERR_LAUNCH : DSX_OK);
}

// ---------------------------------------------------------------------------------------
// emission in depth order: a workgroup owns a range of OUTPUT pairs and walks the blocks of 256
// depth-ordered Gaussians that reach into it; four output pairs to a thread, so the work per
// workgroup is bounded and the stores are contiguous however uneven the tile counts are
// ---------------------------------------------------------------------------------------

// Bound by the issue of vector instructions where a Gaussian has many pairs, so a thread makes four consecutive ones:
// the scan for their owners and the division of the first one's place are paid once, the others advance by one or
// begin a run, and the stores are 16 bytes wide.  18 M pairs of 1 M Gaussians: 89 instructions a pair and 51 us with
// one pair to a thread -> 39; 3.4 M of 3 M Gaussians, most of them out of sight, 27 -> 25.  (1024 workgroups: 29 and 40; 4096: 26 and 40.)
constexpr int kEmitQuad = 4;                        // consecutive outputs of a thread
constexpr int kEmitRound = kEmitQuad * kProjBlock;  // outputs of a workgroup's round
constexpr int kEmitChunkMax = 4096;                 // outputs per workgroup: at most this many ...
constexpr int kEmitWorkgroups = 2048;               // ... and fewer when that leaves less than this many workgroups

// four words at an address that is a multiple of their own size only (the lists may begin anywhere)
template <typename T>
struct __attribute__((packed, aligned(alignof(T)))) Quad
{
    T v[kEmitQuad];
};

// The histograms of two digits (256 words each) from that of one digit of both, where more pairs were found than one digit is taken for.
// (Not where the slots are counted: there it made the counting of 32400 tiles 43 -> 48 us, whose loop the compiler then laid out
// otherwise; as a launch of its own it takes 3 us.)
struct NarrowJob
{
    const uint32_t* wide;
    uint32_t* two; // null: none
    int slots;     // of `wide`; what lies behind them is not counted
    int shift;     // bits of the first digit
};
__device__ __forceinline__ void narrow_digits(const NarrowJob& J, uint32_t* hist, int tid)
{
    __syncthreads();
    for(int j = tid; j < 2 * kBins32; j += kProjBlock)
        hist[j] = 0;
    __syncthreads();
    for(int slot = tid; slot < J.slots; slot += kProjBlock)
    {
        const uint32_t count = J.wide[slot];
        atomicAdd(&hist[slot & ((1 << J.shift) - 1)], count);
        atomicAdd(&hist[kBins32 + (slot >> J.shift)], count);
    }
    __syncthreads();
    for(int j = tid; j < 2 * kBins32; j += kProjBlock)
        J.two[j] = hist[j];
}

// kMasks (lists per bin, SlotT = uint32_t): the high half of a pair's slot word says which tiles of the
// bin the Gaussian's rectangle covers, bit x for the columns and bit 8 + y for the rows of the bin
// (a rectangle is the product of a column range and a row range).  The partition sorts by the low bits
// only and carries the rest along; the blend kernels pick a tile's entries out of its bin's list by
// testing the tile's two bits.  Pairs of negative depth (slot 0, one list for the whole image) carry
// all sixteen bits.
template <typename SlotT, bool kMasks>
__global__ __launch_bounds__(kProjBlock) void emit_ordered_kernel(const uint32_t* __restrict__ order,
                                                                  const uint2* __restrict__ rects_sorted,
                                                                  const uint32_t* __restrict__ block_offsets,
                                                                  int64_t n, int64_t k, int ntx, int shift,
                                                                  SlotT* __restrict__ slots, int32_t* __restrict__ ids,
                                                                  const int32_t* __restrict__ ranges_in,
                                                                  int32_t* __restrict__ ranges_out, int range_count,
                                                                  uint32_t* __restrict__ clear, int64_t clear_words,
                                                                  int chunk, const NarrowJob narrow)
{
    // per Gaussian of the block: x = first output, y = slot of the rectangle's first tile or bin, z = lists in
    // a row of the rectangle (16 bits; bit 31: a negative depth, all pairs go to slot 0), with masks also the
    // rectangle's first column and row (3 bits each) and w = the ones behind its last (16 bits each), all
    // counted from the first bin's
    __shared__ uint4 s_rec[kProjBlock];
    __shared__ uint32_t s_id[kProjBlock];
    __shared__ uint32_t s_total;
    __shared__ __attribute__((aligned(16))) uint32_t wave_tot[kProjBlock / DSX_WAVE];
    __shared__ __attribute__((aligned(16))) uint32_t s_mark[kEmitRound];
    __shared__ __attribute__((aligned(16))) uint32_t s_wave_max[kProjBlock / DSX_WAVE];
    static_assert(kProjBlock == 4 * DSX_WAVE, "four wavefronts per workgroup");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    uint4* const my_marks = reinterpret_cast<uint4*>(s_mark) + tid;
    *my_marks = make_uint4(0u, 0u, 0u, 0u);

    // the tile ranges were derived from the rectangles before any pair existed: hand them out
    for(int j = blockIdx.x * kProjBlock + tid; j < range_count; j += gridDim.x * kProjBlock)
        ranges_out[j] = ranges_in[j];
    // housekeeping for the partition that follows: its counters and look-back statuses start at zero
    for(int64_t j = (int64_t)blockIdx.x * kProjBlock + tid; j < clear_words; j += (int64_t)gridDim.x * kProjBlock)
        clear[j] = 0u;

    // This workgroup's share: outputs [o0, o1).  The work is cut by OUTPUTS, not by Gaussians: a
    // block of 256 near Gaussians can own a hundred thousand pairs and a block of far ones a few
    // hundred, and a workgroup that walked a whole heavy block alone set the kernel's time.
    const int64_t o0 = (int64_t)blockIdx.x * chunk;
    const int64_t o1 = min(o0 + chunk, k);
    if(o0 >= o1) // uniform
    {
        if(narrow.two) // (a workgroup more than there are shares)
            narrow_digits(narrow, reinterpret_cast<uint32_t*>(s_rec), tid);
        return;
    }
    const int64_t blocks = (n + kProjBlock - 1) / kProjBlock;
    // first block of 256 Gaussians (in depth order) whose outputs reach into the share: the largest
    // b with block_offsets[b] <= o0, by a 64-way search (every wavefront does it for itself)
    int64_t first = 0;
    {
        int64_t lo = 0, hi = blocks; // block_offsets[lo] <= o0; the answer lies in [lo, hi)
        while(hi - lo > 1)
        {
            const int64_t step = (hi - lo + 63) / 64;
            const int64_t probe = lo + lane * step;
            const bool ok = probe < hi && (int64_t)block_offsets[probe] <= o0; // true for a prefix of the lanes
            const int reached = __popcll(__ballot(ok)) - 1;                   // lane 0 always holds
            lo += reached * step;
            hi = min(hi, lo + step);
        }
        first = lo;
    }
    for(int64_t blk = first; blk < blocks; ++blk)
    {
        const int64_t base = block_offsets[blk];
        if(base >= o1) // uniform: the share is complete
            break;
        __syncthreads(); // the previous round has finished with the LDS arrays
        const int64_t p = blk * kProjBlock + tid;
        uint32_t count = 0;
        uint4 rec = make_uint4(0u, 0u, 0u, 0u);
        if(p < n)
        {
            // (ntx: lists per row, i.e. bins per row when the lists are binned)
            s_id[tid] = order[p];
            const uint2 r = rects_sorted[p];
            count = list_count(r, shift);
            const uint32_t sx = r.x & 0xffffu, sy = r.x >> 16, w = r.y & 0xffffu, h = (r.y >> 16) & 0x7fffu;
            const bool negative = (r.y >> 31) != 0;
            rec.y = (sy >> shift) * (uint32_t)ntx + (sx >> shift) + 1u;
            rec.z = w;
            if(kMasks)
            {
                const uint32_t x = sx & ((1u << shift) - 1u), y = sy & ((1u << shift) - 1u);
                rec.z = (count ? bin_rect(r, shift).bw : 1u) | (x << 16) | (y << 19);
                rec.w = (x + w) | ((y + h) << 16);
            }
            if(negative)
                rec.z = 0x8000ffffu;
        }
        const uint32_t incl = wave_incl_scan32(count, lane);
        if(lane == 63)
            wave_tot[wave] = incl;
        __syncthreads();
        const uint32_t prefix = sum_of_waves_before<kProjBlock / DSX_WAVE>(wave_tot, wave);
        rec.x = prefix + incl - count;
        s_rec[tid] = rec;
        if(tid == kProjBlock - 1)
            s_total = prefix + incl;
        __syncthreads();

        const int total = (int)s_total, my_start = (int)rec.x; // (fewer than 2^30 pairs in all)
        // the block's outputs that fall into the share: [ja, jb) of its `total`
        const int ja = (int)(max(o0, base) - base);
        const int jb = (int)(min(o1, base + (int64_t)total) - base);
        if(jb <= ja) // uniform (an empty block, or one that ends before the share)
            continue;
        // Which Gaussian owns output j?  Every Gaussian that emits marks the output where its run
        // starts with (its index + 1); the owner of j is the largest mark at or before j, i.e. an
        // inclusive max-scan over the outputs: inside a thread's four, over the wavefront (DPP), over the
        // wavefronts and over the rounds (LDS).
        uint32_t carry = 0; // mark of the owner of the last output before the round
        if(ja > 0)          // uniform: the share starts inside the block
        {
            // the last Gaussian whose run starts before ja (starts are monotone in the thread index)
            const uint64_t early = __ballot(count && my_start < ja);
            if(lane == 0)
                s_wave_max[wave] = early ? (uint32_t)(wave * DSX_WAVE + 64 - __builtin_clzll(early)) : 0u;
            __syncthreads();
            carry = max(max(s_wave_max[0], s_wave_max[1]), max(s_wave_max[2], s_wave_max[3]));
            __syncthreads();
        }
        // (rounds begin at a multiple of four of the whole output: a thread's four lie in one 16-byte word of it)
        for(int j0 = ja - (int)((base + ja) & (kEmitQuad - 1)); j0 < jb; j0 += kEmitRound) // uniform
        {
            if(count && my_start >= j0 && my_start < j0 + kEmitRound)
                s_mark[my_start - j0] = (uint32_t)tid + 1u;
            __syncthreads();
            const uint4 m = *my_marks;
            *my_marks = make_uint4(0u, 0u, 0u, 0u); // ready for the next round (and the next block)
            const uint32_t mark[kEmitQuad] = {m.x, m.y, m.z, m.w};
            const uint32_t incl_max = wave_incl_max_scan(max(max(m.x, m.y), max(m.z, m.w)));
            if(lane == 63)
                s_wave_max[wave] = incl_max;
            __syncthreads();
            const uint4 wm = *reinterpret_cast<const uint4*>(s_wave_max);
            // the owner of the output before this thread's first (wave_shr:1: the lane below)
            uint32_t owner = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl_max, 0x138, 0xf, 0xf, false);
            owner = max(max(owner, carry), max(wave > 0 ? wm.x : 0u, max(wave > 1 ? wm.y : 0u, wave > 2 ? wm.z : 0u)));
            carry = max(carry, max(max(wm.x, wm.y), max(wm.z, wm.w)));
            const int j = j0 + kEmitQuad * tid;
            if(j < jb)
            {
                Quad<SlotT> slot4;
                Quad<int32_t> id4;
                uint32_t rx = 0, ry = 0, w = 0, row = 0; // the place in the rectangle, its width, slots of the rows before
#pragma unroll
                for(int i = 0; i < kEmitQuad; ++i)
                {
                    owner = max(owner, mark[i]);
                    const uint4 rec_i = s_rec[(owner - 1u) & (kProjBlock - 1)]; // (every output of the share has an owner)
                    if(i == 0)
                    {
                        const uint32_t r = (uint32_t)j - rec_i.x;
                        w = rec_i.z & 0xffffu;
                        // r / w by a float reciprocal (r < 2^24 tiles per Gaussian), corrected by one step
                        ry = (uint32_t)((float)r * __builtin_amdgcn_rcpf((float)w));
                        if(ry * w > r)
                            --ry;
                        else if((ry + 1) * w <= r)
                            ++ry;
                        rx = r - ry * w;
                        row = ry * (uint32_t)ntx;
                    }
                    else
                    {
                        ++rx;
                        const bool next_row = rx == w, next_run = mark[i] != 0;
                        rx = next_row || next_run ? 0u : rx;
                        ry = next_run ? 0u : ry + (next_row ? 1u : 0u);
                        row = next_run ? 0u : row + (next_row ? (uint32_t)ntx : 0u);
                        w = rec_i.z & 0xffffu;
                    }
                    uint32_t slot = row + rec_i.y + rx;
                    if(kMasks)
                    {
                        // the rectangle's columns and rows inside this bin, as bit ranges [lo, hi)
                        const int side = 1 << shift, x0 = (int)(rx << shift), y0 = (int)(ry << shift);
                        const int xlo = max((int)((rec_i.z >> 16) & 7u) - x0, 0), ylo = max((int)((rec_i.z >> 19) & 7u) - y0, 0);
                        const int xhi = min((int)(rec_i.w & 0xffffu) - x0, side), yhi = min((int)(rec_i.w >> 16) - y0, side);
                        slot |= ((1u << 16) << xhi) - ((1u << 16) << xlo) + ((1u << 24) << yhi) - ((1u << 24) << ylo);
                    }
                    slot = (int)rec_i.z < 0 ? (kMasks ? 0xffff0000u : 0u) : slot;
                    slot4.v[i] = (SlotT)slot;
                    id4.v[i] = (int32_t)s_id[(owner - 1u) & (kProjBlock - 1)];
                }
                const int64_t out = base + j;
                if(j >= ja && j + kEmitQuad <= jb)
                {
                    *reinterpret_cast<Quad<SlotT>*>(slots + out) = slot4;
                    *reinterpret_cast<Quad<int32_t>*>(ids + out) = id4;
                }
                else
                {
#pragma unroll
                    for(int i = 0; i < kEmitQuad; ++i)
                        if(j + i >= ja && j + i < jb)
                        {
                            slots[out + i] = slot4.v[i];
                            ids[out + i] = id4.v[i];
                        }
                }
            }
            // (the next round's marks are written after this round's reads of s_wave_max: the
            // barrier after them orders both)
        }
    }
}

// tile slots 0..num_tiles fit 16 bits for every image up to 65534 tiles (4K has 32400)
static bool slots_are_u16(int num_tiles)
{
    return num_tiles + 1 <= 65535;
}

// binned: the slot words are 32 bits (slot in the low half, the tile mask in the high half) and the
// sorted ones end in the caller's buffer, behind the ids
ListsWorkspace lists_workspace(int64_t n, int64_t k, int num_tiles, bool binned)
{
    auto align = [](size_t x) { return (x + 255) & ~(size_t)255; };
    ListsWorkspace w;
    const size_t slot_bytes = (binned || !slots_are_u16(num_tiles)) ? 4 : 2;
    const bool wide = one_wide_digit(slot_bits(num_tiles), n, k, binned);
    w.passes = partition_digits(slot_bits(num_tiles), wide).passes;
    size_t off = 0;
    w.slots_a = off;
    off = align(off + (size_t)k * slot_bytes);
    w.slots_b = off;
    off = align(off + (binned ? 0 : (size_t)k * slot_bytes));
    w.ids_alt = off;
    off = align(off + (size_t)k * 4);
    w.sort = off;
    off += sort32_workspace(k, slot_bits(num_tiles), sort32_tile_keys(k), wide).bytes;
    w.bytes = align(off);
    return w;
}

// num_tiles: lists that the pairs are partitioned into (tiles, or bins when the lists are binned: kMasks)
template <typename SlotT, bool kMasks>
static int tile_lists_impl(const dsx_camera& cam, int64_t n, int64_t k, int num_tiles, const void* order,
                           int32_t* sorted_ids, int32_t* ranges, void* workspace, hipStream_t stream)
{
    const OrderLayout o = order_layout(n, cam.image_width, cam.image_height, camera_bin(cam));
    const char* obase = static_cast<const char*>(order);
    const ListGrid lg = list_grid(cam);
    const RangesLayout rl = ranges_layout(lg);
    // what the depth order left ready: everything but the part that the blend forward writes
    const int ready_words = rl.ready;
    if(k <= 0)
    {
        // no pairs: the ranges are all zero (and no tile is occupied)
        int rc = launch_fill_u32(reinterpret_cast<uint32_t*>(ranges), ready_words, 0u, stream);
        if(rc == DSX_OK && lg.shift)
            rc = launch_fill_u32(reinterpret_cast<uint32_t*>(ranges) + rl.header, 1, (uint32_t)lg.shift, stream);
        if(rc == DSX_OK && lg.shift)
            rc = launch_fill_u32(reinterpret_cast<uint32_t*>(ranges) + rl.last_tile, 1, 0xffffffffu, stream);
        return rc;
    }
    const ListsWorkspace w = lists_workspace(n, k, num_tiles, kMasks);
    const int bits = slot_bits(num_tiles);
    const bool wide = one_wide_digit(bits, n, k, kMasks);
    char* base = static_cast<char*>(workspace);
    uint32_t* ids_final = reinterpret_cast<uint32_t*>(sorted_ids);
    uint32_t* ids_other = reinterpret_cast<uint32_t*>(base + w.ids_alt);
    // ping-pong parity: start so that the last pass lands the ids in the caller's buffer (and, for
    // binned lists, the slot words with their masks right behind them)
    const bool even = (w.passes % 2) == 0;
    uint32_t* vals_a = even ? ids_final : ids_other;
    uint32_t* vals_b = even ? ids_other : ids_final;
    SlotT* slots_final = kMasks ? reinterpret_cast<SlotT*>(ids_final + k) : reinterpret_cast<SlotT*>(base + w.slots_b);
    SlotT* slots_other = reinterpret_cast<SlotT*>(base + w.slots_a);
    SlotT* slots_a = (kMasks && even) ? slots_final : slots_other;
    SlotT* slots_b = (kMasks && even) ? slots_other : slots_final;
    int rc = DSX_OK;
    const Sort32Workspace sw = sort32_workspace(k, bits, sort32_tile_keys(k), wide);
    const uint32_t* counts = reinterpret_cast<const uint32_t*>(obase + o.slot_hist);
    NarrowJob narrow = {};
    if(!wide && wide_digit_most(bits, n, kMasks) > 0) // (counted for one digit before the number of pairs was known)
    {
        static_assert(kWideBits <= 2 * kBits32 && sizeof(uint4) * kProjBlock >= 2 * kBins32 * 4, "two digits, in the records' memory");
        narrow = {counts, reinterpret_cast<uint32_t*>(base + w.sort + sw.hist), num_tiles + 1, digits32(bits).shift[1]};
        counts = narrow.two;
    }
    // (what lies behind the histogram starts at zero)
    const size_t clear_from = narrow.two ? sw.counters : sw.hist;
    {
        DSX_TIMED("emit_ordered_kernel", stream);
        // outputs per workgroup: a multiple of 256 between 256 and kEmitChunkMax
        const int64_t want = (k + kEmitWorkgroups - 1) / kEmitWorkgroups;
        const int chunk = (int)min((int64_t)kEmitChunkMax, ((want + kProjBlock - 1) / kProjBlock) * kProjBlock);
        hipLaunchKernelGGL((emit_ordered_kernel<SlotT, kMasks>), dim3((unsigned)((k + chunk - 1) / chunk) + (narrow.two ? 1 : 0)),
                           dim3(kProjBlock), 0, stream, reinterpret_cast<const uint32_t*>(obase + o.ids_a),
                           reinterpret_cast<const uint2*>(obase + o.rects_sorted),
                           reinterpret_cast<const uint32_t*>(obase + o.block_sums), n, k,
                           lg.shift ? lg.nbx : lg.ntx, lg.shift, slots_a, reinterpret_cast<int32_t*>(vals_a),
                           reinterpret_cast<const int32_t*>(obase + o.ranges), ranges, ready_words,
                           reinterpret_cast<uint32_t*>(base + w.sort + clear_from), (int64_t)((sw.bytes - (clear_from - sw.hist)) / 4), chunk, narrow);
    }
    DSX_LAUNCH_CHECK();
    SlotT* ko;
    uint32_t* vo;
    // per-tile lists: the sorted slots themselves are not needed (the ranges are known already);
    // binned lists: they are kept for their masks
    rc = DSX_ERR_RUNTIME;
    auto partition = [&](auto items, auto digit_bits) {
        return sort32_passes<SlotT, kSortThreads32, decltype(items)::value, false, decltype(digit_bits)::value>(
            k, bits, slots_a, vals_a, slots_b, vals_b, false, kMasks, base + w.sort, "onesweep32_kernel<tile partition>", stream, &ko, &vo,
            nullptr, nullptr, counts);
    };
#define DSX_PARTITION_ITEMS(ITEMS)                                                                                     \
    case ITEMS:                                                                                                        \
        rc = !wide        ? partition(std::integral_constant<int, ITEMS>(), std::integral_constant<int, kBits32>())    \
             : bits == 9  ? partition(std::integral_constant<int, ITEMS>(), std::integral_constant<int, 9>())          \
             : bits == 10 ? partition(std::integral_constant<int, ITEMS>(), std::integral_constant<int, 10>())         \
                          : partition(std::integral_constant<int, ITEMS>(), std::integral_constant<int, kWideBits>());  \
        break
    switch(sort32_items(k))
    {
        DSX_PARTITION_ITEMS(1);
        DSX_PARTITION_ITEMS(2);
        DSX_PARTITION_ITEMS(3);
        DSX_PARTITION_ITEMS(4);
        DSX_PARTITION_ITEMS(6);
        DSX_PARTITION_ITEMS(8);
        DSX_PARTITION_ITEMS(kSortItemsMax32);
    }
#undef DSX_PARTITION_ITEMS
    if(rc)
        return rc;
    if(kMasks && ko != slots_final)
        return DSX_ERR_RUNTIME;
    return vo == ids_final ? DSX_OK : DSX_ERR_RUNTIME;
}

// order: buffer of order_layout(n) after launch_depth_order.  Writes sorted_ids[k] and the ready part
// of ranges (ranges_layout: per-tile ranges and, for binned lists, the last occupied tile and the
// bins' ranges).
int launch_tile_lists(const dsx_camera& cam, int64_t n, int64_t k, const void* order, int32_t* sorted_ids,
                      int32_t* ranges, void* workspace, hipStream_t stream)
{
    const ListGrid lg = list_grid(cam);
    const int num_tiles = lg.lists();
    if(k >= (1ll << 30))
        return DSX_ERR_TOO_LARGE;
    if(n <= 0)
        k = 0;
    if(lg.shift)
    {
        if(num_tiles + 1 > 65535) // (the slot shares its word with the 16-bit mask)
            return DSX_ERR_TOO_LARGE;
        return tile_lists_impl<uint32_t, true>(cam, n, k, num_tiles, order, sorted_ids, ranges, workspace, stream);
    }
    if(slots_are_u16(num_tiles))
        return tile_lists_impl<uint16_t, false>(cam, n, k, num_tiles, order, sorted_ids, ranges, workspace, stream);
    return tile_lists_impl<uint32_t, false>(cam, n, k, num_tiles, order, sorted_ids, ranges, workspace, stream);
}

} // namespace dsx
