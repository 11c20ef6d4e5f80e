// Register-resident tree dedispersion on gfx950: stage 1, and stage 2 with any subband search.
//
// Reference semantics: ReferenceTree (src_lib/ReferenceTree.cpp:120-345) as applied by
// ReferenceDedisperser sophistication 1 (src_lib/ReferenceDedisperser.cpp:388-450):
//   pass r pairs rows e = fout*2^(r+1) + dmb and o = e + 2^r (in place, bit-reversed DM):
//     e <- c*(x_e[t - L] + x_o[t]),  o <- c*(x_e[t - L - 1] + x_o[t]),  L = bitrev(dmb, r).
//
// Factorization (the same identity that splits the full tree into stage 1 and stage 2):
// a rank-DD tree over rows i = h*2^K1 + l (K1 + K2 = DD) equals
//   phase A: 2^K2 independent rank-K1 trees over l (one per h),
//   a delay of (2^K2 - 1 - h) * bitrev(j, K1) samples on row (h, j), j = phase-A output row,
//   phase B: 2^K1 independent rank-K2 trees over h (one per j); final row = h'*2^K1 + j.
// The floating-point operations are exactly those of the direct tree, so results are
// bit-identical.
//
// Subbands. Stage 2 takes K2 = pf_rank, the peak finder's rank, so the rows of one phase-B tree
// are the 2^pf_rank level-0 bands at one coarse DM pf_dm = bitrev(j, K1): every stream of that
// DM (ReferenceTree.cpp:142-287) is a value of this tree. Band pfs of level 0 is row pfs before
// the first pass; band pfs of level l is an output pair of pass l - 1 (pfs even), or a butterfly
// of two neighbouring groups before that pass (pfs odd, "staggered"). A band that ends at
// row fhi comes out (2^pf_rank - fhi) * pf_dm samples late, the phase delay of its last row:
// that is the final lag the reference applies to the stream (ReferenceTree.cpp:42-54), so
// streams need no further delay.
//
// Mapping: one workgroup per tree instance sweeps the chunk in tiles of U = 96 samples (rank 8:
// 64), one sub-tree's rows per wave in registers. Both phases work in windows: lane = two
// consecutive samples, and the first OVA = 2^K1 (phase A) or OV = 2^K2 (phase B) samples of a
// window come before the tile and only feed the lags. So there are no histories to hold or to
// select from, and a shift by L and L + 1 together takes 3 lane moves for two samples instead of
// 4. A window of 96 samples fills 48 to 56 of 64 lanes (rank 1 to rank 7), one of 64 no more than 40.
//   Rank 8 has LDS for tiles of 64 to 80 samples only; there phase A holds lane = one sample,
// with lanes t < L taking the previous tile's values (tree_regs.hpp).
// Between the phases a row goes through an LDS line that holds its last lag + OV samples and the
// current tile; phase A appends at the end, phase B reads the OV + U samples at the start and
// moves the line down by U. The lines persist across chunks in an HBM state buffer, with the last OVA input samples of stage 1 (stage
// 2 finds its own in the ring, whose rows are OVA samples longer) or rank 8's histories.
//
// A chunk that is no multiple of U ends in a smaller tile (a multiple of 32 samples): its loads
// stay inside the chunk, its stores stop at the chunk's end, and the lines move down by its
// length.
//
// Bounded by the round trips of a tile (row loads, two barriers, LDS lines; waves wait half of
// their time), then by VALU issue (62% busy in float16), not by bytes: rank 7 runs at 4.2-4.6 TB/s in float32, 2.9-3.2 in
// float16. 16 beams of 16384 channels x 2048 samples, stages 1 and 2 (rank 7): float16 0.83 and
// 0.86 ms with tiles of 64 and phase-A histories, 0.69 and 0.75 ms now; float32 0.99 and 0.95,
// 1.00 and 0.90 ms. Rank 8 (4 beams of 65536 channels, float16) with histories 1.05 and 1.08 ms,
// in windows and tiles of 64 1.16 and 1.26, of 80 1.07 and 1.14; its subband stage 2 1.26, 1.48
// and 1.61 ms (rows of 80 16-bit samples start inside 64-byte blocks).
// No kernel spills, and none calls a function: with the line offsets in a recursive constexpr
// function the compiler called it at run time, in the tile loop, with all live registers saved
// around it (rank 8 stage 1 2.10 ms, with a table 1.06 ms; the kernels that kept both phases'
// histories in registers 2.61 ms). Subband stage 2 with the passes after the first emission in
// LDS, a barrier after each: rank 8 4.25 ms, rank 6 with 34 multiplets 0.58 -> 0.18 ms.
//
// Segments: with few tree instances the chunk is cut into nseg runs of tiles (blockIdx.z).
// Phase B keeps nothing from tile to tile, so a later segment only has to run phase A over the
// tiles that fill its lines (and histories) before its own (WARM tiles).

#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"
#include "tree_regs.hpp"

namespace pirate_amd {

namespace {

using namespace treg;

constexpr int cmin(int a, int b) { return (a < b) ? a : b; }

template<int DD>
struct RegDims {
    static constexpr int D = 1 << DD;
    static constexpr int K1 = DD / 2, K2 = (DD + 1) / 2;
    static constexpr int NRA = 1 << K1, NRB = 1 << K2;      // rows of a phase-A / phase-B sub-tree
    // waves per workgroup: rank 8 one sub-tree per wave and phase in 16 waves, lower ranks 8 waves
    static constexpr int NW = (DD >= 8) ? 16 : cmin(8, cmin(NRA, NRB));
    static constexpr int SA = NRB / NW;                     // phase-A sub-trees per wave
    static_assert(NRA == NW, "one phase-B sub-tree per wave");
    // Phase A in windows, as phase B, or (rank 8) one sample per lane with histories: where LDS
    // keeps the tile at 64 samples, 16 more in each window cost more than the histories (figures
    // at the top).
    static constexpr bool HIST = DD >= 8;
    static constexpr int S = HIST ? 1 : 2;                  // phase-A samples per lane
    // samples per tile: for 2 samples per lane as many as 64 lanes and two workgroups' lines in
    // LDS take. A multiple of 32, as are chunks, so that a chunk's last tile is one as well.
    static constexpr int U = HIST ? 64 : 96;
    static constexpr int OVA = (K1 > 0 && !HIST) ? NRA : 0, OV = NRB;    // window samples before the tile
    static constexpr int WLA = (OVA + U) / S, WL = (OV + U) / 2;         // lanes of a window
    static constexpr int T2 = NRB * (NRB - 1) / 2;
    static constexpr int SUMB = NRA * (NRA - 1) / 2;         // sum of bitrev(j) over j
    static constexpr int NRES = (T2 * SUMB + D * OV + 1) & ~1;     // saved line samples (an odd number at rank 2)
    // and the histories, or stage 1's last input samples
    static constexpr int nstate(bool stage2) { return NRES + (HIST ? NRB * Sub<K1>::NST : stage2 ? 0 : D * OVA); }
    static constexpr int LMAX = (NRB - 1) * (NRA - 1);
    // tiles that fill a segment's lines (lag + OV samples), with histories from outputs that no
    // longer depend on the zeros it started with (the first NRA - 1 samples do)
    static constexpr int WARM = (LMAX + OV + (HIST ? NRA - 1 : 0) + U - 1) / U;
    static_assert(WLA <= 64 && WL <= 64, "a window fits a wave");
    static_assert(HIST || (NRES % 2 == 0 && nstate(false) % 2 == 0), "saved input samples are read and written in aligned pairs");

    // Line (h, j): even(lag) + OV + U floats, j-major, so that every line starts 8-byte aligned.
    static constexpr int LINE0 = OV + U;
    static constexpr int G(int h) { return h * (NRB - 1) - h * (h - 1) / 2; }    // sum of (NRB-1-h') over h' < h
    // start of the lines of j (a table: a function of j, even constexpr, is called at run time
    // where j only becomes constant by unrolling)
    struct Starts {
        int v[NRA + 1];
    };
    static constexpr Starts starts()
    {
        Starts t{};
        for (int j = 0; j < NRA; j++)
            t.v[j + 1] = t.v[j] + NRB * LINE0 + brev_c(j, K1) * T2 + (brev_c(j, K1) & 1) * (NRB / 2);
        return t;
    }
    static constexpr Starts CQ = starts();
    __host__ __device__ static constexpr int lag(int h, int bj) { return (NRB - 1 - h) * bj; }
    // start of line (h, j) within the lines of j; bj = bitrev(j, K1)
    __host__ __device__ static constexpr int line(int h, int bj) { return h * LINE0 + bj * G(h) + (bj & 1) * ((h + 1) >> 1); }
    // + what lanes past a window read
    static constexpr int DL_FLOATS = ((CQ.v[NRA] + ((LMAX + OV > 128) ? 192 : 128) + 3) / 4) * 4;
    static constexpr int LDS_BYTES = 4 * DL_FLOATS;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
    // saved samples of line (h, j): lag + OV floats, j-major
    __device__ static int res(int h, int j, int bj, int sumb) { return T2 * sumb + bj * G(h) + (j * NRB + h) * OV; }
};

// Two consecutive samples per lane.
struct Two {
    float x, y;
};

// v of lane - a (a = 0..NRB/2, compile-time after unrolling). Lanes below a get what feeds no
// output (the window's first samples).
__device__ __forceinline__ float lane_up(float v, int a, int lane)
{
    if (a == 0)
        return v;
    if (a == 1)
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));    // wave_shr:1
    return __int_as_float(__builtin_amdgcn_ds_bpermute(((lane - a) & 63) << 2, __float_as_int(v)));
}

// c*(e delayed by L + o) and c*(e delayed by L + 1 + o).
__device__ __forceinline__ void butterfly(const Two &e, const Two &o, int L, int lane, Two &out0, Two &out1)
{
    const int a = L >> 1;
    Two d0, d1;
    if (L & 1) {
        d0.x = lane_up(e.y, a + 1, lane);
        d0.y = lane_up(e.x, a, lane);
        d1.x = lane_up(e.x, a + 1, lane);
        d1.y = d0.x;
    } else {
        d0.x = lane_up(e.x, a, lane);
        d0.y = lane_up(e.y, a, lane);
        d1.x = lane_up(e.y, a + 1, lane);
        d1.y = d0.x;
    }
    out0.x = kRsqrt2 * (d0.x + o.x);
    out0.y = kRsqrt2 * (d0.y + o.y);
    out1.x = kRsqrt2 * (d1.x + o.x);
    out1.y = kRsqrt2 * (d1.y + o.y);
}

// A wave-uniform value that the compiler must take as new: offsets formed from it are computed
// where they are used (scalar arithmetic), not once per launch for all rows in registers that
// the tile loop does not have.
__device__ __forceinline__ int fresh(int x)
{
    asm volatile("" : "+s"(x));
    return x;
}

// Reads the windows at the start of the lines of rows h0 .. h0 + NL - 1 of a phase-B sub-tree
// and moves these lines down by sh samples (U, or the chunk's last samples: even). All by one
// wave, whose LDS instructions execute in order; a line's loads are issued before the stores that
// may overwrite what they read, and the loads of NL lines are in flight together. Of every line
// the first lag(h0) + OV samples are stored, under one mask: the lag falls with h, and what that
// writes past a line's own lag + OV samples lies in its tile, which phase A writes next.
template<int DD, int NL, bool READ>
__device__ __forceinline__ void take_lines(float *lj, int h0, int b, int lane, int sh, Two *v)
{
    using F = RegDims<DD>;
    static_assert((NL - 1) * (F::NRA - 1) <= F::U, "lag(h0) + OV samples of a line lie within it");
    const int keep = F::lag(h0, b) + F::OV;
    constexpr bool LONG = F::LMAX + F::OV > 128;
    const bool lng = LONG && keep > 128;      // wave-uniform
    float2 s0[NL], s1[NL], *q[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        q[i] = reinterpret_cast<float2 *>(lj + fresh(F::line(h0 + i, b))) + lane;
        if constexpr (READ) {
            const float2 w = *q[i];
            v[i].x = w.x;
            v[i].y = w.y;
        }
        s0[i] = q[i][sh / 2];
    }
    if (lng) {
#pragma unroll
        for (int i = 0; i < NL; i++)
            s1[i] = q[i][sh / 2 + 64];
    }
    __builtin_amdgcn_wave_barrier();
    if (2 * lane < keep) {
#pragma unroll
        for (int i = 0; i < NL; i++)
            *q[i] = s0[i];
    }
    if (lng && 128 + 2 * lane < keep) {
#pragma unroll
        for (int i = 0; i < NL; i++)
            q[i][64] = s1[i];
    }
    __builtin_amdgcn_wave_barrier();
}

// S (1 or 2) consecutive samples as loaded, at any element alignment.
template<typename Tst, int S>
struct RawS {
    raw_st<Tst> v;
    __device__ __forceinline__ void load(const Tst *p) { v = ld_raw(p); }
    __device__ __forceinline__ void set(const Tst *p, const Tst *) { v = ld_raw(p); }
};
template<>
struct RawS<float, 2> {
    typedef float V __attribute__((ext_vector_type(2), aligned(4)));
    V v;
    __device__ __forceinline__ void load(const float *p) { v = *reinterpret_cast<const V *>(p); }
    __device__ __forceinline__ void set(const float *p, const float *q) { v = V{*p, *q}; }
    __device__ __forceinline__ Two get() const { return Two{v.x, v.y}; }
};
template<typename T16>
struct RawTwo16 {
    typedef unsigned V __attribute__((aligned(2)));
    unsigned v;
    __device__ __forceinline__ void load(const T16 *p) { v = *reinterpret_cast<const V *>(p); }
    __device__ __forceinline__ void set(const T16 *p, const T16 *q) { v = ld_raw(p) | (ld_raw(q) << 16); }
    __device__ __forceinline__ Two get() const { return Two{from_raw<T16>(v & 0xffffu), from_raw<T16>(v >> 16)}; }
};
template<> struct RawS<__half, 2> : RawTwo16<__half> { };
template<> struct RawS<__hip_bfloat16, 2> : RawTwo16<__hip_bfloat16> { };

// Element offset of a ring row held by lane k: up to 2^32 elements per beam.
__device__ __forceinline__ unsigned lane_offset(int v, int k) { return unsigned(__builtin_amdgcn_readlane(v, k)); }

__device__ __forceinline__ int rowlen_of(const Stage1Args &) { return 0; }
__device__ __forceinline__ int rowlen_of(const Stage2Args &a) { return a.rowlen; }
__device__ __forceinline__ int nband_of(const Stage1Args &, int) { return 0; }
__device__ __forceinline__ int nband_of(const Stage2Args &a, int lev) { return a.nband[lev]; }

template<typename Tst, int DD, bool STAGE2, typename Args>
__device__ __forceinline__ void reg_tree_body(const Args &a)
{
    using F = RegDims<DD>;
    using SA_ = Sub<F::K1>;
    constexpr int D = F::D, U = F::U;
    extern __shared__ __align__(16) float lbuf[];

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tr = blockIdx.x, b = blockIdx.y;
    const long gbeam = long(a.beam0) + b;

    const long chunk = launch_chunk(a);

    // this segment's tiles
    const int ntiles = (a.Tp + U - 1) / U;
    const int first = int(blockIdx.z) * ntiles / a.nseg, end = (int(blockIdx.z) + 1) * ntiles / a.nseg;
    const int start = blockIdx.z ? first - F::WARM : 0;       // >= 0: the host checks it

    const StateBlocks blocks = a.chunk_dev ? a.blocks_of(chunk) : a.blocks;
    float *st = a.state + b * a.state_bstride + long(tr) * F::nstate(STAGE2);
    const float *rd = st + blocks.rd * a.B * a.state_bstride;
    float *wr = st + blocks.wr * a.B * a.state_bstride;

    // this wave's phase-B sub-tree j: bitrev(j), its lines, and sum of bitrev(j') over j' < j
    const int j = wid, bj = __builtin_amdgcn_readfirstlane(bitrev_dev(j, F::K1));
    int line0 = 0, sumb = 0;
    for (int k = 0; k < j; k++) {
        const int bk = bitrev_dev(k, F::K1);
        line0 += F::NRB * F::LINE0 + bk * F::T2 + (bk & 1) * (F::NRB / 2);
        sumb += bk;
    }
    line0 = __builtin_amdgcn_readfirstlane(line0);
    sumb = __builtin_amdgcn_readfirstlane(sumb);
    if (start == 0) {
        for (int h = 0; h < F::NRB; h++) {
            float *p = lbuf + line0 + F::line(h, bj);
            const float *r = rd + F::res(h, j, bj, sumb);
            for (int q = lane; q < F::lag(h, bj) + F::OV; q += 64)
                p[q] = r[q];
        }
    }

    float ha[F::HIST ? F::SA : 1][F::HIST ? SA_::NH : 1];
    if constexpr (F::HIST) {
#pragma unroll
        for (int s = 0; s < F::SA; s++) {
            if (start == 0) {
                load_hist<F::K1>(ha[s], rd + F::NRES + (wid + s * F::NW) * SA_::NST, lane);
            } else {
#pragma unroll
                for (int i = 0; i < SA_::NH; i++)
                    ha[s][i] = 0.0f;
            }
        }
    }

    // The wave's ring rows, one per lane: element offset, position and capacity (32-bit, checked
    // on the host). Stage 1 writes the rows hp*NRA + j (lane hp) of its phase-B sub-tree, at the
    // position of the next tile; stage 2 reads the rows of its phase-A sub-trees (lane s*NRA + l) at
    // their lag, from the start of the next tile's window. A tile that no row wraps in takes one
    // lane read per row and scalar addresses.
    unsigned roff;
    int rpos, rcap;
    {
        long rr, t = chunk * a.Tp + start * U;
        if constexpr (!STAGE2) {
            rr = long(tr) * D + cmin(lane, F::NRB - 1) * F::NRA + j;
        } else {
            const int i = cmin(lane, F::SA * F::NRA - 1);
            rr = (long((wid + (i / F::NRA) * F::NW) * F::NRA + i % F::NRA) << a.amb) + tr;
            t -= a.row_lag[rr] + F::OVA;
        }
        const long cap = a.ring.row_cap[rr];
        roff = unsigned(a.ring.row_off[rr]);
        rpos = int(ring_pos(t, cap));
        rcap = int(cap);
    }
    auto advance = [&](int n) {
        rpos += n;
        rpos -= (rpos >= rcap) ? rcap : 0;
    };

    const Tst *src;    // stage 1: this tree's input rows; stage 2: the beam's ring
    Tst *dst;          // stage 1: the beam's ring; stage 2: the beam's peak-finder rows
    if constexpr (!STAGE2) {
        src = reinterpret_cast<const Tst *>(a.in) + long(b) * a.in_bstride + long(tr) * D * a.Tp;
        dst = reinterpret_cast<Tst *>(a.ring.base) + gbeam * a.ring.bstride;
    } else {
        src = reinterpret_cast<const Tst *>(a.ring.base) + gbeam * a.ring.bstride;
        dst = reinterpret_cast<Tst *>(a.sb) + gbeam * a.sb_bstride + a.tpad;
    }

    // Phase-A windows of tile t0, issued one tile ahead and kept as loaded until phase A converts
    // them. Lanes past the window (or the chunk) load its last samples. Stage 1 clamps what lies
    // before the chunk to its start: phase A takes the saved samples there.
    RawS<Tst, F::S> xa[F::SA][F::NRA];
    auto load_a = [&](int t0) {
        const int wlen = F::OVA + min(U, a.Tp - t0);           // a capacity holds a whole window
        const int i = min(F::S * lane, wlen - F::S);
        if constexpr (!STAGE2) {
            const unsigned tb = unsigned(max(t0 - F::OVA + i, 0)) * unsigned(sizeof(Tst));
#pragma unroll
            for (int s = 0; s < F::SA; s++) {
                const int h = fresh(wid + s * F::NW);
#pragma unroll
                for (int l = 0; l < F::NRA; l++) {
                    const Tst *row = src + long(h * F::NRA + l) * a.Tp;
                    xa[s][l].load(reinterpret_cast<const Tst *>(reinterpret_cast<const char *>(row) + tb));
                }
            }
        } else {
            const unsigned tb = unsigned(i) * unsigned(sizeof(Tst));
            const int q = int(roff + unsigned(rpos));
            const unsigned long long wrap = __ballot(rpos + wlen > rcap);
            auto load_row = [&](int s, int l) {
                const Tst *row = src + lane_offset(q, s * F::NRA + l);
                xa[s][l].load(reinterpret_cast<const Tst *>(reinterpret_cast<const char *>(row) + tb));
            };
            if (wrap == 0) {
#pragma unroll
                for (int s = 0; s < F::SA; s++)
#pragma unroll
                    for (int l = 0; l < F::NRA; l++)
                        load_row(s, l);
            } else {
                // About one tile in two: some row wraps. Float32 loads only such rows sample by
                // sample (stage 2 0.933 -> 0.904 ms); 16-bit types do it for all rows, since
                // with both ways the halves of a pair make the compiler wait row by row
                // (0.752 -> 0.939 ms), and so does rank 8, for want of registers.
                constexpr bool ALL = sizeof(Tst) == 2 || F::S == 1;
#pragma unroll
                for (int s = 0; s < F::SA; s++)
#pragma unroll
                    for (int l = 0; l < F::NRA; l++) {
                        const int k = s * F::NRA + l;
                        if (ALL || ((wrap >> k) & 1)) {
                            const int cap = __builtin_amdgcn_readlane(rcap, k);
                            const Tst *row = src + lane_offset(int(roff), k);
                            const int q0 = __builtin_amdgcn_readlane(rpos, k) + i, q1 = q0 + 1;
                            xa[s][l].set(row + (q0 - ((q0 >= cap) ? cap : 0)), row + (q1 - ((q1 >= cap) ? cap : 0)));
                            if constexpr (!ALL)
                                asm volatile("");        // keeps the branches' loads (and their addresses) apart
                        } else {
                            load_row(s, l);
                        }
                    }
                asm volatile("");
            }
            advance(U);
        }
    };

    // Tile t0 of nv samples: U, or what is left of the chunk (a multiple of 32).
    using Full = std::integral_constant<int, U>;
    auto tile_step = [&](int t0, bool warm, auto nv_) {
        const int nv = nv_;
#pragma unroll
        for (int s = 0; s < F::SA; s++) {
            const int h = fresh(wid + s * F::NW);
            if constexpr (F::HIST) {
                float x[F::NRA];
#pragma unroll
                for (int l = 0; l < F::NRA; l++)
                    x[l] = from_raw<Tst>(xa[s][l].v);
                sub_passes<F::K1>(x, ha[s], lane);
#pragma unroll
                for (int jj = 0; jj < F::NRA; jj++) {
                    constexpr int K1 = F::K1;
                    const int b1 = brev_c(jj, K1);
                    lbuf[F::CQ.v[jj] + F::line(h, b1) + F::lag(h, b1) + F::OV + lane] = x[jj];
                }
            } else {
                Two x[F::NRA];
#pragma unroll
                for (int l = 0; l < F::NRA; l++)
                    x[l] = xa[s][l].get();
                if constexpr (!STAGE2 && F::OVA > 0) {
                    // the input samples before the chunk, and the chunk's last ones for the next
                    if (t0 == 0 && lane < F::OVA / 2) {
#pragma unroll
                        for (int l = 0; l < F::NRA; l++) {
                            const float2 y = *reinterpret_cast<const float2 *>(rd + F::NRES + (h * F::NRA + l) * F::OVA + 2 * lane);
                            x[l] = Two{y.x, y.y};
                        }
                    }
                    const int k = 2 * lane - nv;
                    if (t0 + nv == a.Tp) {
                        // in place, a chunk of one tile writes where other lanes have just read
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    }
                    if (t0 + nv == a.Tp && k >= 0 && k < F::OVA) {
#pragma unroll
                        for (int l = 0; l < F::NRA; l++)
                            *reinterpret_cast<float2 *>(wr + F::NRES + (h * F::NRA + l) * F::OVA + k) = make_float2(x[l].x, x[l].y);
                    }
                }
#pragma unroll
                for (int r = 0; r < F::K1; r++) {
                    const int G = 1 << r;
#pragma unroll
                    for (int e0 = 0; e0 < F::NRA; e0 += 2 * G)
#pragma unroll
                        for (int d = 0; d < G; d++) {
                            Two o0, o1;
                            butterfly(x[e0 + d], x[e0 + d + G], brev_c(d, r), lane, o0, o1);
                            x[e0 + d] = o0;
                            x[e0 + d + G] = o1;
                        }
                }
                if (lane >= F::OVA / 2 && lane < F::WLA) {
#pragma unroll
                    for (int jj = 0; jj < F::NRA; jj++) {
                        constexpr int K1 = F::K1;
                        const int b1 = brev_c(jj, K1);
                        float *p = lbuf + fresh(F::CQ.v[jj] + F::line(h, b1) + F::lag(h, b1) + F::OV - F::OVA) + 2 * lane;
                        p[0] = x[jj].x;
                        p[1] = x[jj].y;
                    }
                }
            }
        }
        __syncthreads();
        if (t0 + U < a.Tp)
            load_a(t0 + U);

        float *lj = lbuf + fresh(line0);
        const int b1 = fresh(bj);
        constexpr int NL = cmin(4, F::NRB);
        Two y[F::NRB];
#pragma unroll
        for (int h = 0; h < F::NRB; h += NL) {
            if (warm)
                take_lines<DD, NL, false>(lj, h, b1, lane, nv, y + h);
            else
                take_lines<DD, NL, true>(lj, h, b1, lane, nv, y + h);
        }
        if (warm) {
            if constexpr (!STAGE2)
                advance(U);
            __syncthreads();
            return;
        }

        const bool live = lane >= F::OV / 2 && lane < (F::OV + nv) / 2;
        // stage 2: window lane 0's sample of multiplet 0 of this coarse DM
        Tst *row = nullptr;
        const int rowlen = STAGE2 ? fresh(rowlen_of(a)) : 0;
        if constexpr (STAGE2)
            row = dst + ((long(bitrev_dev(tr, a.amb)) << (DD - F::K2)) + b1) * a.M * rowlen + (t0 - F::OV);
        auto emit = [&](int m, const Two &v) {
            if constexpr (STAGE2)
                st2_st(row + long(m * rowlen) + unsigned(2 * lane), v.x, v.y);
        };
        if constexpr (STAGE2) {
            const int nb = fresh(a.nband[0]);
            if (nb > 0 && live) {
#pragma unroll
                for (int p = 0; p < F::NRB; p++)
                    if (p < nb)
                        emit(p, y[p]);
            }
        }
#pragma unroll
        for (int r = 0; r < F::K2; r++) {
            const int G = 1 << r;                        // rows of a group before the pass
            const int nb = STAGE2 ? fresh(nband_of(a, r + 1)) : 0;
            if constexpr (STAGE2) {
                if (nb > 1) {                            // odd bands: groups p and p + 1
                    const int m0 = fresh(a.mband[r + 1]);
#pragma unroll
                    for (int p = 1; p + 1 < F::NRB / G; p += 2)
                        if (p < nb) {
#pragma unroll
                            for (int x = 0; x < G; x++) {
                                const int L = brev_c(x, r);
                                Two o0, o1;
                                butterfly(y[p * G + x], y[(p + 1) * G + x], L, lane, o0, o1);
                                const int m = m0 + p * 2 * G + 2 * L;
                                if (live) {
                                    emit(m, o0);
                                    emit(m + 1, o1);
                                }
                            }
                        }
                }
            }
#pragma unroll
            for (int g = 0; g < F::NRB / (2 * G); g++)
#pragma unroll
                for (int x = 0; x < G; x++) {
                    const int e = g * 2 * G + x, L = brev_c(x, r);
                    Two o0, o1;
                    butterfly(y[e], y[e + G], L, lane, o0, o1);
                    y[e] = o0;
                    y[e + G] = o1;
                }
            if constexpr (STAGE2) {
                if (nb > 0 && live) {                    // even bands: the pass's outputs
                    const int m0 = fresh(a.mband[r + 1]);
#pragma unroll
                    for (int g = 0; g < F::NRB / (2 * G); g++)
                        if (2 * g < nb) {
#pragma unroll
                            for (int x = 0; x < G; x++) {
                                const int e = g * 2 * G + x, L = brev_c(x, r);
                                const int m = m0 + g * 4 * G + 2 * L;
                                emit(m, y[e]);
                                emit(m + 1, y[e + G]);
                            }
                        }
                }
            }
        }
        if constexpr (!STAGE2) {
            // Ring positions and capacities are multiples of 32: a lane's two samples never
            // part. The lane reads stay outside the branch on live: what is formed inside it is
            // formed for live lanes only, and lane 0 is not one.
            if (!__any(rpos + nv > rcap)) {
                const int q = int(roff + unsigned(rpos));
                unsigned qs[F::NRB];
#pragma unroll
                for (int hp = 0; hp < F::NRB; hp++)
                    qs[hp] = lane_offset(q, hp);
                if (live) {
#pragma unroll
                    for (int hp = 0; hp < F::NRB; hp++)
                        st2_st(dst + (long(qs[hp]) - F::OV) + unsigned(2 * lane), y[hp].x, y[hp].y);
                }
            } else {
#pragma unroll
                for (int hp = 0; hp < F::NRB; hp++) {
                    const int cap = __builtin_amdgcn_readlane(rcap, hp);
                    Tst *row = dst + lane_offset(int(roff), hp);
                    int q = __builtin_amdgcn_readlane(rpos, hp) + 2 * lane - F::OV;
                    q -= (q >= cap) ? cap : 0;
                    if (live)
                        st2_st(row + q, y[hp].x, y[hp].y);
                }
            }
            advance(nv);
        }
        __syncthreads();
    };

    load_a(start * U);
    const int nfull = a.Tp / U;
    for (int it = start; it < min(end, nfull); it++)
        tile_step(it * U, it < first, Full{});
    if (end > nfull)
        tile_step(nfull * U, false, a.Tp - nfull * U);

    if (blockIdx.z + 1 == gridDim.z) {
        if constexpr (F::HIST) {
#pragma unroll
            for (int s = 0; s < F::SA; s++)
                save_hist<F::K1>(ha[s], wr + F::NRES + (wid + s * F::NW) * SA_::NST, lane, (a.Tp - 1) % U + 1);
        }
        for (int h = 0; h < F::NRB; h++) {
            const float *p = lbuf + line0 + F::line(h, bj);
            float *r = wr + F::res(h, j, bj, sumb);
            for (int q = lane; q < F::lag(h, bj) + F::OV; q += 64)
                r[q] = p[q];
        }
    }
}

template<typename Tst, int DD>
__global__ void __launch_bounds__(RegDims<DD>::NW * 64) __attribute__((amdgpu_waves_per_eu((DD >= 4) ? 4 : 2)))
k_stage1(Stage1Args a)
{
    reg_tree_body<Tst, DD, false>(a);
}

template<typename Tst, int DD>
__global__ void __launch_bounds__(RegDims<DD>::NW * 64) __attribute__((amdgpu_waves_per_eu((DD >= 4) ? 4 : 2)))
k_stage2(Stage2Args a)
{
    reg_tree_body<Tst, DD, true>(a);
}

}  // namespace


// Dynamic LDS above 64 KB (ranks 7 and 8) must be allowed per kernel; gfx950 allows 160 KB.
static void allow_lds(const void *fn, int bytes)
{
    if (bytes > 65536)
        (void) hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

// Time segments: a segment of n tiles runs n + WARM; workgroups run in rounds of as many as fit
// on the chip (256 CUs, 16 waves and 160 KB of LDS each), and a round costs about kStart tiles
// besides (launch, state). Takes the power of two with the shortest sum. One beam of rank 10
// (32 instances x 22 tiles): stages 1 and 2 54 and 64 us in one segment, 13 and 12 us in 16; from some
// 500 instances on, one segment.
template<typename F>
static int tree_nseg(long ninst, int Tp)
{
    constexpr int kStart = 2;
    constexpr long slots = 256L * cmin(16 / F::NW, 160 * 1024 / F::LDS_BYTES);
    const int ntiles = (Tp + F::U - 1) / F::U;
    int best = 1;
    long cost = 0;
    for (int n = 1; n == 1 || (ntiles / n >= cmin(F::WARM, ntiles) && n <= ntiles); n *= 2) {
        const long rounds = (ninst * n + slots - 1) / slots;
        const long c = rounds * ((ntiles + n - 1) / n + (n > 1 ? F::WARM : 0) + kStart);
        if (n == 1 || c < cost) {
            best = n;
            cost = c;
        }
    }
    return best;
}

// Calls f(RegDims<dd>()), dd = 1..8; r for other ranks.
template<typename R, typename F>
static R for_rank(int dd, R r, F f)
{
    switch (dd) {
        case 1: return f(RegDims<1>());
        case 2: return f(RegDims<2>());
        case 3: return f(RegDims<3>());
        case 4: return f(RegDims<4>());
        case 5: return f(RegDims<5>());
        case 6: return f(RegDims<6>());
        case 7: return f(RegDims<7>());
        case 8: return f(RegDims<8>());
        default: return r;
    }
}

int tree_segments(int dd, long ninst, int Tp)
{
    return for_rank(dd, 1, [&](auto d) { return tree_nseg<decltype(d)>(ninst, Tp); });
}

long tree_state_nelts(int dd, bool stage2)
{
    return for_rank(dd, 0L, [&](auto d) { return long(d.nstate(stage2)); });
}

int tree_overlap(int dd)
{
    return for_rank(dd, 0, [](auto d) { return int(d.OVA); });
}

template<int DD, typename Args>
static void launch_tree(void (*k)(Args), const Args &a, hipStream_t st)
{
    using F = RegDims<DD>;
    allow_lds((const void *) k, F::LDS_BYTES);
    hipLaunchKernelGGL(k, dim3(1 << a.amb, a.B, a.nseg), dim3(F::NW * 64), F::LDS_BYTES, st, a);
}

template<typename Tst>
static void launch_stage1_t(const Stage1Args &a, hipStream_t st)
{
    switch (a.dd) {
#define PDD_T(DDV) case DDV: launch_tree<DDV>(k_stage1<Tst, DDV>, a, st); break;
        PDD_T(1) PDD_T(2) PDD_T(3) PDD_T(4) PDD_T(5) PDD_T(6) PDD_T(7) PDD_T(8)
#undef PDD_T
        default: break;
    }
}

template<typename Tst>
static void launch_stage2_t(const Stage2Args &a, hipStream_t st)
{
    switch (a.dd) {
#define PDD_T(DDV) case DDV: launch_tree<DDV>(k_stage2<Tst, DDV>, a, st); break;
        PDD_T(1) PDD_T(2) PDD_T(3) PDD_T(4) PDD_T(5) PDD_T(6) PDD_T(7) PDD_T(8)
#undef PDD_T
        default: break;
    }
}

void launch_stage1(Dtype dt, const Stage1Args &a, hipStream_t st)
{
    switch (dt) {
        case Dtype::float32: launch_stage1_t<float>(a, st); break;
        case Dtype::float16: launch_stage1_t<__half>(a, st); break;
        case Dtype::bfloat16: launch_stage1_t<__hip_bfloat16>(a, st); break;
    }
}

void launch_stage2(Dtype dt, const Stage2Args &a, hipStream_t st)
{
    switch (dt) {
        case Dtype::float32: launch_stage2_t<float>(a, st); break;
        case Dtype::float16: launch_stage2_t<__half>(a, st); break;
        case Dtype::bfloat16: launch_stage2_t<__hip_bfloat16>(a, st); break;
    }
}

}  // namespace pirate_amd
