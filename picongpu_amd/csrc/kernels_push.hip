// Fused field gather + particle push + moveParticle + Esirkepov deposit.
//
// One workgroup per supercell (the reference's KernelMoveAndMarkParticles,
// particles/Particles.kernel:169-273, and KernelComputeCurrent,
// fields/FieldJ.kernel:51-107). The E/B tile of the supercell plus the
// interpolation margins is staged in LDS; particles of all species in the
// launch are streamed as coalesced SoA slot reads; each particle's current
// is accumulated into an int64 fixed-point J tile in LDS (order independent)
// that is flushed once to HBM. Launches run over a checkerboard of
// supercells whose J tiles do not overlap, so the flush is a plain
// read-add-write in a fixed phase order.
#include <type_traits>

#include "pic_device.hpp"
#include "pic_kernels.hpp"
#include "pic_shift_common.hpp"

namespace pic {

__device__ __forceinline__ int wrapIdx(int v, int n) {
    v = v < 0 ? v + n : v;
    return v >= n ? v - n : v;
}

constexpr int kPushThreads = kPushThreadsPerBlock;
constexpr int kPushWaves = kPushThreads / 64;

// t / D for 0 <= t < N by one 24-bit multiplication; the compiler's form for
// a general int needs the high half of a 32-bit product, a quarter-rate
// instruction
template <int D, int N>
constexpr bool divSmallExact() {
    for (int t = 0; t < N; ++t)
        if (((t * ((65536 + D - 1) / D)) >> 16) != t / D) return false;
    return true;
}
template <int D, int N>
__device__ __forceinline__ int divSmall(int t) {
    static_assert(divSmallExact<D, N>(), "the reciprocal is too short for this range");
    return (int)(__umul24((unsigned)t, (65536 + D - 1) / D) >> 16);
}

// element t of a box of X x Y x Z elements (x fastest) as coordinates
template <int X, int Y, int Z>
__device__ __forceinline__ void boxCoords(int t, int& x, int& y, int& z) {
    constexpr int N = ((X * Y * Z + kPushThreads - 1) / kPushThreads) * kPushThreads;
    int const row = divSmall<X, N>(t);
    x = t - row * X;
    z = divSmall<Y, N>(row);
    y = row - z * Y;
}

// A particle whose move changes its shifted cell on some axis needs the
// general Esirkepov form (up to (SUPP+1)^2*SUPP cells per component); the rest
// need SUPP^2*(SUPP-1). The push deposits the latter at once and queues the
// former per wave: lane l holds queued item l in A (items 64..127 in B), and
// a full A is deposited by all 64 lanes together. An item is one word: the
// particle's slot, its tile cell and its species in the launch. The deposit
// reads the particle's new state back (its lines were written a few
// iterations ago) and forms its velocity and move from it, the values the
// push formed: the unfused deposit does the same. Keeping the state in the
// queue instead took 16 registers of every wave for the whole loop, and with
// them the kernel spilled.
static_assert(kMaxFrames * SCV <= 1 << 16, "a slot takes 16 bits");
__device__ __forceinline__ uint32_t slowItem(int slot, int cx, int cy, int cz, int species) {
    return (uint32_t)slot | ((uint32_t)cx << 16) | ((uint32_t)cy << 20) | ((uint32_t)cz << 24) |
           ((uint32_t)species << 28);
}

// Append the items of the lanes with `slow` set after the P queued ones
// (wave-uniform P). Every lane of the wave calls it: the ds_permute moves
// slow lanes to queue positions P.. and the other lanes to the free ones, a
// permutation of the 64 lanes.
__device__ __forceinline__ void queueSlow(bool slow, uint32_t mine, uint32_t& A, uint32_t& B, int& P) {
    unsigned long long const m = __ballot(slow);
    int const k = __popcll(m);
    if (k == 0) return;
    int const lane = threadIdx.x & 63;
    int const below = __popcll(m & laneMaskLt());
    int const dst = (P + (slow ? below : k + (lane - below))) & 63;
    int const off = (lane - P) & 63;
    uint32_t const r = (uint32_t)__builtin_amdgcn_ds_permute(dst << 2, (int)mine);
    if (off < k && lane >= P) A = r;
    if (off < k && lane < P) B = r;
    P += k;
}

// the deposit of the queued particle `item` of supercell sc
template <int SUPP, class TG>
__device__ __forceinline__ void depositQueued(unsigned long long* __restrict__ sJ, const PushArgs& a, int sc,
                                              uint32_t item, const DepositConsts& dk) {
    static_assert(SCX + Esirkepov<SUPP>::lowerMargin < 16 && PIC_MAX_SPECIES <= 4, "fields of an item");
    Vec3 pos{0.0f, 0.0f, 0.0f}, mom{0.0f, 0.0f, 0.0f};
    float mass = 0.0f, charge = 0.0f;
    int const species = (int)(item >> 28);
    for (int s = 0; s < a.nsp; ++s) {  // uniform; a lane loads in its species' round
        const SpeciesDev& S = a.sp[s];
        if (species != s) continue;
        size_t const gidx = slotBase(S, sc) + (item & 0xffffu);
        pos = Vec3{S.pos[0][gidx], S.pos[1][gidx], S.pos[2][gidx]};
        mom = Vec3{S.mom[0][gidx], S.mom[1][gidx], S.mom[2][gidx]};
        float const w = S.w[gidx];
        mass = S.mass * w;
        charge = S.charge * w;
    }
    Vec3 const vel = velocityOf(mom, mass);
    Esirkepov<SUPP>::template depositGeometry<TG, true>(sJ, (item >> 16) & 15, (item >> 20) & 15, (item >> 24) & 15,
                                                        Esirkepov<SUPP>::geometry(pos, vel, dk), charge, dk);
}

// leavers of one species the epilogue keeps in LDS (slot and exchange code);
// a supercell with more takes the lists in global memory
constexpr int kLeaverListLds = 2048;

// LDS bytes of one supercell's work: the E/B tile (or the epilogue's
// scratch), then the int64 J tile
template <int SUPP, int MODE>
struct PushLds {
    using TG = JTileGeom<Esirkepov<SUPP>::lowerMargin, Esirkepov<SUPP>::upperMargin>;
    static constexpr int EB_ELEMS = MODE == 2 ? 1 : EBTile<SUPP>::total();
    static constexpr int J_ELEMS = MODE == 0 ? 1 : TG::total();
    static constexpr int EB_BYTES = ((EB_ELEMS * 4 + 15) / 16) * 16;
    static constexpr int EPI_BYTES =
        MODE == 2 ? 0
                  : (kPushMaxIters * kPushWaves + 1) * 4 + kPushWaves * kNumDirs * 4 + (int)sizeof(GroupScratch) +
                        kLeaverListLds * 4;
    // 16-byte multiple: the int64 J tile that follows needs 8-byte aligned LDS addresses
    static constexpr int LO_BYTES = (((EB_BYTES > EPI_BYTES ? EB_BYTES : EPI_BYTES) + 15) / 16) * 16;
    // odd support: a byte per wave, whether it staged a non-finite node
    static constexpr int BAD_AT = LO_BYTES + J_ELEMS * 8;
    static constexpr int BYTES = BAD_AT + (MODE != 2 && EBTile<SUPP>::ODD ? kPushWaves : 0);
};

// J += the tile's component C. A thread's J values are loaded together, then
// added and stored; an element that adds nothing (zero, or beyond an open
// border) loads J's first cell instead and stores nothing. inside: the tile
// lies in the box on every axis (uniform).
template <class TG, int C, int DLO>
__device__ __forceinline__ void flushComponent(const PushArgs& a, const unsigned long long* sJ, int ox, int oy, int oz,
                                               bool inside) {
    constexpr int VOL = TG::vol(C);
    constexpr int NU = (VOL + kPushThreads - 1) / kPushThreads;
    float* const J = a.J[C];
    float add[NU], old[NU];
    size_t gi[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        int const t = threadIdx.x + u * kPushThreads;
        long long const acc = fixedTileValue(sJ[TG::off(C) + (t < VOL ? t : 0)]);
        int tx, ty, tz;
        boxCoords<TG::ext(C, 0), TG::ext(C, 1), TG::ext(C, 2)>(t, tx, ty, tz);
        int gx = ox - DLO + tx, gy = oy - DLO + ty, gz = oz - DLO + tz;
        bool adds = t < VOL && acc != 0;
        if (!inside) {
            adds = adds && !(a.g.open && outsideOpen(a.g, gx, gy, gz));
            gx = wrapIdx(gx, a.g.nx);
            gy = wrapIdx(gy, a.g.ny);
            gz = wrapIdx(gz, a.g.nz);
        }
        size_t const at = (size_t)gx + (size_t)a.g.nx * ((size_t)gy + (size_t)a.g.ny * gz);
        gi[u] = adds ? at : 0;
        add[u] = adds ? (float)((double)acc * a.jinv) : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) old[u] = J[gi[u]];
#pragma unroll
    for (int u = 0; u < NU; ++u)
        if (add[u] != 0.0f) J[gi[u]] = old[u] + add[u];
}

// The shift's staging of one species from its leaver bits, with the leaver
// list in LDS (L <= kLeaverListLds entries): the records of the leavers go to
// the outbox grouped by exchange code (ascending slot inside a code), the
// offset table to outOff, and the supercell is compacted as stageSC does.
// `pre`: per (iteration, wave) entry the number of leavers before it. The
// same orders as groupLeavers and stageSC; the list never leaves the CU, so
// a supercell waits for three memory round trips (the codes, the records,
// the moved particles) instead of ten.
__device__ void stageFromBits(const SpeciesDev& S, int sc, int n, int iters, uint32_t bits, int L, const uint32_t* pre,
                              GroupScratch& g, uint32_t* sWaveCnt, uint32_t* sList) {
    int const tid = threadIdx.x;
    int const lane = tid & 63;
    int const wave = tid >> 6;
    size_t const base = slotBase(S, sc);
    uint32_t* const off = S.outOff + (size_t)sc * kOffStride;
    if (L == 0) {  // uniform
        if (tid < kOffStride) off[tid] = 0u;
        return;
    }
    if (tid < kNumDirs) g.cnt[tid] = 0u;
    for (int it = 0; it < iters; ++it) {
        bool const left = (bits >> it) & 1u;
        unsigned long long const m = __ballot(left);
        if (left) sList[pre[it * kPushWaves + wave] + (uint32_t)__popcll(m & laneMaskLt())] = it * kPushThreads + tid;
    }
    __syncthreads();
    for (int k = tid; k < L; k += kPushThreads) {
        uint32_t const slot = sList[k];
        uint32_t const code = (uint32_t)S.mask[base + slot] - 1u;
        sList[k] = slot | (code << 16);
        atomicAdd(&g.cnt[code], 1u);
    }
    __syncthreads();
    if (wave == 0) {  // offsets of the codes 1..26, [27] = L
        uint32_t const c = lane >= 1 && lane < kNumDirs ? g.cnt[lane] : 0u;
        uint32_t const before = waveInclusiveScan(c) - c;
        if (lane < kNumDirs) g.run[lane] = before;
        if (lane < kOffStride) off[lane] = before;
    }
    for (int c0 = 0; c0 < L; c0 += kPushThreads) {
        int const k = c0 + tid;
        uint32_t const e = k < L ? sList[k] : 0u;
        int const code = (int)(e >> 16);
        size_t const from = base + (e & 0xffffu);
        float4 r0, r1;
        if (code != 0) {
            r0 = make_float4(S.pos[0][from], S.pos[1][from], S.pos[2][from], S.mom[0][from]);
            r1 = make_float4(S.mom[1][from], S.mom[2][from], S.w[from], __int_as_float((int)S.cell[from]));
        }
        for (int j = tid; j < kNumDirs * kPushWaves; j += kPushThreads) sWaveCnt[j] = 0u;
        __syncthreads();
        int myRank = 0;
        unsigned long long pending = __ballot(code != 0);
        while (pending) {
            int const leader = __ffsll((long long)pending) - 1;
            int const kc = __shfl(code, leader);
            unsigned long long const same = __ballot(code == kc);
            if (code == kc) myRank = __popcll(same & laneMaskLt());
            if (lane == 0) sWaveCnt[wave * kNumDirs + kc] = (uint32_t)__popcll(same);
            pending &= ~same;
        }
        __syncthreads();
        if (code != 0) {
            uint32_t r = g.run[code] + (uint32_t)myRank;
            for (int w = 0; w < wave; ++w) r += sWaveCnt[w * kNumDirs + code];
            S.outbox[2 * (base + r)] = r0;
            S.outbox[2 * (base + r) + 1] = r1;
        }
        if (c0 + kPushThreads < L) {
            __syncthreads();
            if (tid > 0 && tid < kNumDirs) {
                uint32_t add = 0;
                for (int w = 0; w < kPushWaves; ++w) add += sWaveCnt[w * kNumDirs + tid];
                g.run[tid] += add;
            }
            __syncthreads();
        }
    }
    __syncthreads();  // every leaver record has been read before its slot is overwritten
    int const nn = n - L;
    int run = 0;
    for (int it = nn / kPushThreads; it < iters; ++it) {
        int const i = it * kPushThreads + tid;
        bool const stays = i >= nn && i < n && !((bits >> it) & 1u);
        int total;
        int const r = blockRank<kPushWaves>(stays, sWaveCnt, &total);
        if (stays) {
            size_t const dst = base + (sList[run + r] & 0xffffu);
            copyParticle(S, dst, base + i);
            S.mask[dst] = 1;
        }
        run += total;
    }
    for (int i = nn + tid; i < n; i += kPushThreads) S.mask[base + i] = 0;
    if (tid == 0) S.count[sc] = (uint32_t)nn;
}

// The work of one supercell `sc` of the simulation described by `a`; every
// thread of the workgroup calls it.
template <int SUPP, int PUSHER, int MODE, bool EMZ = false, bool DAMP = false>
__device__ __forceinline__ void pushDepositSC(const PushArgs& a, int sc, unsigned char* smem) {
    constexpr int GLO = SUPP / 2;          // FieldToParticleInterpolation.hpp:49
    constexpr int GUP = (SUPP + 1) / 2;    // FieldToParticleInterpolation.hpp:50
    constexpr int GX = SCX + GLO + GUP, GY = SCY + GLO + GUP, GZ = SCZ + GLO + GUP;
    constexpr int GV = GX * GY * GZ;
    // The J tile is the supercell plus the reference's deposit margins. In
    // the fused form the deposit runs in the frame of the particle's new
    // cell, which may lie one cell outside the supercell, but the cells it
    // touches still lie within those margins of the particle's old cell: its
    // path starts inside the old cell and moves less than one cell per axis
    // (the host requires float(c*dt)/cell < 1).
    constexpr int DLO = Esirkepov<SUPP>::lowerMargin;
    constexpr int UPM = Esirkepov<SUPP>::upperMargin;
    using TG = JTileGeom<DLO, UPM>;
    constexpr int EB_ELEMS = MODE == 2 ? 1 : EBTile<SUPP>::total();
    constexpr int J_ELEMS = MODE == 0 ? 1 : TG::total();

    // One LDS buffer: the E/B tile, then the J tile. After the particle loop
    // the E/B tile is dead and its space holds the epilogue's scratch.
    constexpr int LO_BYTES = PushLds<SUPP, MODE>::LO_BYTES;
    static_assert(LO_BYTES % 16 == 0, "J tile must be 16-byte aligned");
    static_assert(EB_ELEMS == PushLds<SUPP, MODE>::EB_ELEMS && J_ELEMS == PushLds<SUPP, MODE>::J_ELEMS, "LDS plan");
    float* const sEB = reinterpret_cast<float*>(smem);
    unsigned long long* const sJ = reinterpret_cast<unsigned long long*>(smem + LO_BYTES);
    uint32_t* const sPre = reinterpret_cast<uint32_t*>(smem);
    uint32_t* const sWaveCnt = sPre + kPushMaxIters * kPushWaves + 1;
    GroupScratch& sGroup = *reinterpret_cast<GroupScratch*>(sWaveCnt + kPushWaves * kNumDirs);
    uint32_t* const sList = reinterpret_cast<uint32_t*>(&sGroup + 1);
    uint8_t* const sBad = reinterpret_cast<uint8_t*>(smem + PushLds<SUPP, MODE>::BAD_AT);

    if (halted(a.g)) return;  // uniform: a later step of an overflowed simulation
    int const sx = sc % a.g.nscx;
    int const sy = (sc / a.g.nscx) % a.g.nscy;
    int const sz = sc / (a.g.nscx * a.g.nscy);
    int const ox = sx * SCX, oy = sy * SCY, oz = sz * SCZ;
    // opaque, so that a persistent workgroup's loop over supercells does not
    // keep the staging's node offsets in registers (they spilled)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    __builtin_assume(tid >= 0 && tid < kPushThreads);

    int total = 0;
    for (int s = 0; s < a.nsp; ++s) total += (int)a.sp[s].count[sc];
    if (total == 0) {  // uniform across the workgroup
        if (MODE != 2 && tid < kOffStride) {
            for (int s = 0; s < a.nsp; ++s) a.sp[s].outOff[(size_t)sc * kOffStride + tid] = 0u;
        }
        if (MODE != 0 && a.tileOut && tid == 0) a.tileHeld[sc] = 0u;  // the gather flush passes its tile over
        return;
    }

    // The E/B tile: a thread's node offsets are formed once for the six
    // components, and all its loads are in flight before the first LDS write
    // (a loop of load and write costs a memory latency per round, which a
    // supercell of few particles does not hide). Supercells whose tile lies
    // inside the box skip the wrap.
    if (MODE != 2) {
        using T = EBTile<SUPP>;
        constexpr int NU = (GV + kPushThreads - 1) / kPushThreads;
        bool const inside = ox >= GLO && ox + SCX + GUP <= a.g.nx && oy >= GLO && oy + SCY + GUP <= a.g.ny &&
                            oz >= GLO && oz + SCZ + GUP <= a.g.nz;
        size_t gi[NU];
        bool out[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            int tx, ty, tz;
            boxCoords<GX, GY, GZ>(tid + u * kPushThreads, tx, ty, tz);
            int gx = ox - GLO + tx, gy = oy - GLO + ty, gz = oz - GLO + tz;
            out[u] = false;
            if (!inside) {  // uniform
                out[u] = a.g.open && outsideOpen(a.g, gx, gy, gz);  // fields beyond an open border read zero
                gx = wrapIdx(gx, a.g.nx);
                gy = wrapIdx(gy, a.g.ny);
                gz = wrapIdx(gz, a.g.nz);
            }
            gi[u] = (size_t)gx + (size_t)a.g.nx * ((size_t)gy + (size_t)a.g.ny * gz);
            if (tid + u * kPushThreads >= GV) gi[u] = 0;
        }
        float v[6][NU];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const float* const src = c < 3 ? a.E[c] : a.B[c - 3];
#pragma unroll
            for (int u = 0; u < NU; ++u) v[c][u] = src[gi[u]];
        }
        if (T::ODD) {
            // the sum of all is non-finite if one is (an overflow of finite ones only costs time)
            float sum = 0.0f;
#pragma unroll
            for (int u = 0; u < NU; ++u)
                sum += ((v[0][u] + v[1][u]) + (v[2][u] + v[3][u])) + (v[4][u] + v[5][u]);
            uint8_t const any = __ballot(__builtin_amdgcn_classf(sum, 0x207)) != 0ull ? 1 : 0;  // NaN, -Inf, +Inf
            if ((tid & 63) == 0) sBad[tid >> 6] = any;
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            int tx, ty, tz;
            boxCoords<GX, GY, GZ>(tid + u * kPushThreads, tx, ty, tz);
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                // the component's box of nodes within the common one
                int const x = tx - (GLO - T::lo(c, 0)), y = ty - (GLO - T::lo(c, 1)), z = tz - (GLO - T::lo(c, 2));
                if ((unsigned)x >= (unsigned)T::ext(c, 0) || (unsigned)y >= (unsigned)T::ext(c, 1) ||
                    (unsigned)z >= (unsigned)T::ext(c, 2))
                    continue;
                float const f = out[u] ? 0.0f : v[c][u];
                float* const row = sEB + T::off(c) + (z * T::ext(c, 1) + y) * T::pitch(c);
                if (T::ODD) {
                    row[x] = f;
                    if (T::ext(c, 0) % 2 == 1 && x == T::ext(c, 0) - 1) row[x + 1] = 0.0f;  // the pad
                } else {  // node x in the pairs (x, x+1) and (x-1, x)
                    if (x < T::ext(c, 0) - 1) row[2 * x] = f;
                    if (x > 0) row[2 * x - 1] = f;
                }
            }
        }
    }
    if (MODE != 0) {
        static_assert(MODE == 0 || J_ELEMS % 2 == 0, "two tile elements per store");
        for (int t = tid; t < J_ELEMS / 2; t += kPushThreads) reinterpret_cast<ulonglong2*>(sJ)[t] = make_ulonglong2(0ull, 0ull);
    }
    __syncthreads();
    // the same in every lane: not 0 when the tile holds a non-finite node (odd
    // support; read here, first needed after the particle's loads)
    uint32_t badNodes = 0u;
    if (MODE != 2 && EBTile<SUPP>::ODD) {
        static_assert(kPushWaves == 8, "a byte per wave");
        uint2 const b = *reinterpret_cast<const uint2*>(sBad);
        badNodes = b.x | b.y;
    }

    DepositConsts dk;
    dk.cell[0] = a.cell[0];
    dk.cell[1] = a.cell[1];
    dk.cell[2] = a.cell[2];
    dk.rcell[0] = a.rcell[0];
    dk.rcell[1] = a.rcell[1];
    dk.rcell[2] = a.rcell[2];
    dk.rvol = a.rvol;
    dk.inv_vdt = a.inv_vdt;
    dk.jscale = a.jscale;

    // whether a particle of this supercell can end in a damping area (a move
    // is less than a cell per axis): the others skip the exchange loop
    bool dampSC = false;
    if (DAMP && a.damp.axes) {
        int const org[3] = {ox, oy, oz}, ext[3] = {SCX, SCY, SCZ};
#pragma unroll
        for (int d = 0; d < 3; ++d)
            if ((a.damp.axes >> d) & 1)
                dampSC = dampSC || org[d] - 1 < a.damp.lo[d] || org[d] + ext[d] >= a.damp.hi[d];
    }

    uint32_t qA = 0u, qB = 0u;
    int queued = 0;  // wave-uniform
    uint32_t leaveBits = 0u;
    for (int s = 0; s < a.nsp; ++s) {
        const SpeciesDev& S = a.sp[s];
        int const n = (int)S.count[sc];
        size_t const base = slotBase(S, sc);
        leaveBits = 0u;  // bit `it`: the particle of iteration `it` left the supercell (it < kPushMaxIters)
        int const iters = (n + kPushThreads - 1) / kPushThreads;  // uniform across the workgroup
        // the last species runs one iteration more, without particles, that drains the queue
        bool const lastSpecies = s == a.nsp - 1;
        for (int it = 0; it < iters + (MODE == 1 && !EMZ && lastSpecies ? 1 : 0); ++it) {
            int const i = it * kPushThreads + tid;
            bool slow = false;
            uint32_t mine = 0u;
            if (i < n) {
                size_t const gidx = base + i;
                Vec3 const pos{S.pos[0][gidx], S.pos[1][gidx], S.pos[2][gidx]};
                Vec3 mom{S.mom[0][gidx], S.mom[1][gidx], S.mom[2][gidx]};
                float w = S.w[gidx];
                int const lidx = S.cell[gidx];
                int const lx = lidx % SCX, ly = (lidx / SCX) % SCY, lz = lidx / (SCX * SCY);
                float const mass = S.mass * w;     // attribute::getMass (GetMass.hpp:40-44)
                float charge = S.charge * w;       // attribute::getCharge (GetCharge.hpp:45-66)
                if (MODE != 2) {
                    WeightTerms const terms = weightTerms<PUSHER>(mass, charge);
                    GatherWeights<SUPP> const gw(pos, lx, ly, lz);
                    Vec3 e{gather1<SUPP, 0>(sEB, gw), gather1<SUPP, 1>(sEB, gw), gather1<SUPP, 2>(sEB, gw)};
                    Vec3 b{gather1<SUPP, 3>(sEB, gw), gather1<SUPP, 4>(sEB, gw), gather1<SUPP, 5>(sEB, gw)};
                    if constexpr (EBTile<SUPP>::ODD)
                        if (badNodes) gatherStencil<SUPP>(sEB, pos, lx, ly, lz, e, b);
                    Vec3 vel;
                    if (PUSHER == PIC_PUSHER_VAY)
                        pushVay(e, b, mom, vel, mass, charge, terms);
                    else if (PUSHER == PIC_PUSHER_HIGUERA_CARY)
                        pushHigueraCary(e, b, mom, vel, mass, charge, terms);
                    else
                        pushBoris(e, b, mom, vel, mass, charge, terms);
                    float p[3] = {pos.x, pos.y, pos.z};
                    // the move in cells; Esirkepov forms the same quotients (Esirkepov.hpp:82)
                    float dp[3] = {divExact(vel.x, dk.rcell[0]), divExact(vel.y, dk.rcell[1]),
                                   divExact(vel.z, dk.rcell[2])};
                    p[0] += dp[0];
                    p[1] += dp[1];
                    p[2] += dp[2];
                    int dir[3], newIdx, newMask;
                    moveParticle(p, lidx, dir, newIdx, newMask);
                    if (S.reflect) {  // the species' reflecting borders (boundary::apply after the push)
                        int cellNow[3] = {ox + lx + dir[0], oy + ly + dir[1], oz + lz + dir[2]};
                        int const nGrid[3] = {a.g.nx, a.g.ny, a.g.nz};
                        if (reflectParticle(nGrid, S.reflect, cellNow, p, mom, vel, dir, dp))
                            cellAfterMove(lidx, dir, newIdx, newMask);
                    }
                    if (DAMP && dampSC) {
                        // the absorbing boundary's PML damping, exchange by exchange
                        // (+x, -x, +y, -y, +z, -z); the deposit stage then takes the
                        // velocity and charge of the damped particle. One loop, not
                        // unrolled, with the axis' values selected (no indexed local
                        // arrays, which the compiler would move to LDS)
                        int const c0 = ox + lx + dir[0], c1 = oy + ly + dir[1], c2 = oz + lz + dir[2];
                        bool any = false;
                        if (!(a.g.open && outsideOpen(a.g, c0, c1, c2))) {
#pragma unroll 1
                            for (int e = 0; e < 6; ++e) {
                                int const d = e >> 1;
                                if (!((a.damp.axes >> d) & 1) || ((S.reflect >> d) & 1)) continue;
                                int const cn = d == 0 ? c0 : (d == 1 ? c1 : c2);
                                bool const inArea = (e & 1) == 0 ? cn >= a.damp.hi[d] : cn < a.damp.lo[d];
                                if (!inArea) continue;
                                float const pd = d == 0 ? p[0] : (d == 1 ? p[1] : p[2]);
                                float const cs = d == 0 ? a.cell[0] : (d == 1 ? a.cell[1] : a.cell[2]);
                                pmlDamp(a.damp, d, cn, pd, S.mass, cs, mom, w);
                                any = true;
                            }
                        }
                        if (any) {
                            S.w[gidx] = w;
                            charge = S.charge * w;
                            vel = velocityOf(mom, S.mass * w);
                            dp[0] = divExact(vel.x, dk.rcell[0]);
                            dp[1] = divExact(vel.y, dk.rcell[1]);
                            dp[2] = divExact(vel.z, dk.rcell[2]);
                        }
                    }
                    S.pos[0][gidx] = p[0];
                    S.pos[1][gidx] = p[1];
                    S.pos[2][gidx] = p[2];
                    S.mom[0][gidx] = mom.x;
                    S.mom[1][gidx] = mom.y;
                    S.mom[2][gidx] = mom.z;
                    if ((dir[0] | dir[1] | dir[2]) != 0) S.cell[gidx] = (uint16_t)newIdx;
                    if (newMask >= 2) S.mask[gidx] = (uint8_t)newMask;
                    leaveBits |= (newMask >= 2 ? 1u : 0u) << (it & (kPushMaxIters - 1));
                    // a particle leaving through an open border is absorbed by the
                    // boundary before the reference's deposit stage sees it
                    if (MODE == 1 && !(a.g.open && outsideOpen(a.g, ox + lx + dir[0], oy + ly + dir[1], oz + lz + dir[2]))) {
                        int const cx = lx + dir[0] + DLO, cy = ly + dir[1] + DLO, cz = lz + dir[2] + DLO;
                        Vec3 const np{p[0], p[1], p[2]};
                        if (EMZ) {
                            EmZ<SUPP>::template depositDp<TG>(sJ, cx, cy, cz, np, dp, charge, dk);
                        } else {
                            typename Esirkepov<SUPP>::Geometry G;
                            if (Esirkepov<SUPP>::stayGeometry(np, dp, G)) {
                                Esirkepov<SUPP>::template depositStay<TG>(sJ, cx, cy, cz, G, charge, dk);
                            } else {
                                slow = true;
                                mine = slowItem(i, cx, cy, cz, s);
                            }
                        }
                    }
                } else {
                    Vec3 const vel = velocityOf(mom, mass);
                    if (EMZ)
                        EmZ<SUPP>::template deposit<TG>(sJ, lx + DLO, ly + DLO, lz + DLO, pos, vel, charge, dk);
                    else
                        Esirkepov<SUPP>::template deposit<TG>(sJ, lx + DLO, ly + DLO, lz + DLO, pos, vel, charge,
                                                                      dk);
                }
            }
            if (MODE == 1 && !EMZ) {
                queueSlow(slow, mine, qA, qB, queued);
                if (queued >= 64 || (it == iters && queued > 0)) {
                    // the queued particles' stores by other lanes of this wave come first
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if ((int)(tid & 63) < queued) depositQueued<SUPP, TG>(sJ, a, sc, qA, dk);
                    qA = qB;
                    queued = queued > 64 ? queued - 64 : 0;
                }
            }
        }
        // (the last species' bits stay in the register)
        if (MODE != 2 && !lastSpecies) S.leaveBits[(size_t)sc * kPushThreads + tid] = leaveBits;
    }
    __syncthreads();

    if (MODE != 0 && a.tileOut) {
        // one launch for every supercell: the tile is left for the gather
        // flush as the floats the flush would add, zero where it adds
        // nothing (adding a zero would change nothing either: J never holds
        // -0, its sums start at +0 and round to nearest)
        for (int t = tid; t < J_ELEMS; t += kPushThreads) {
            long long const acc = fixedTileValue(sJ[t]);
            a.tileOut[(size_t)sc * J_ELEMS + t] = acc == 0 ? 0.0f : (float)((double)acc * a.jinv);
        }
        if (tid == 0) a.tileHeld[sc] = 1u;
    } else if (MODE != 0) {
        bool const inside = ox >= DLO && ox + SCX + UPM <= a.g.nx && oy >= DLO && oy + SCY + UPM <= a.g.ny &&
                            oz >= DLO && oz + SCZ + UPM <= a.g.nz;
        flushComponent<TG, 0, DLO>(a, sJ, ox, oy, oz, inside);
        flushComponent<TG, 1, DLO>(a, sJ, ox, oy, oz, inside);
        flushComponent<TG, 2, DLO>(a, sJ, ox, oy, oz, inside);
    }

    // Epilogue: the leavers from the per-thread bits, in slot order; in a full
    // step staged for the shift (outbox records, compaction of the supercell),
    // else as the leaver lists of the stage calls.
    if (MODE != 2) {
        for (int s = 0; s < a.nsp; ++s) {
            const SpeciesDev& S = a.sp[s];
            int const n = (int)S.count[sc];
            int const iters = (n + kPushThreads - 1) / kPushThreads;
            int const wave = tid >> 6;
            size_t const base = slotBase(S, sc);
            int L = 0;
            __syncthreads();
            if (iters <= kPushMaxIters) {
                uint32_t const bits =
                    s == a.nsp - 1 ? leaveBits : S.leaveBits[(size_t)sc * kPushThreads + tid];
                // leavers per (iteration, wave) entry, entries in slot order
                for (int it = 0; it < iters; ++it) {
                    unsigned long long const m = __ballot((bits >> it) & 1u);
                    if ((tid & 63) == 0) sPre[it * kPushWaves + wave] = (uint32_t)__popcll(m);
                }
                __syncthreads();
                if (wave == 0) {  // exclusive prefix, four entries per lane
                    constexpr int PER = kPushMaxIters * kPushWaves / 64;
                    int const entries = iters * kPushWaves;
                    uint32_t c[PER], sum = 0;
#pragma unroll
                    for (int e = 0; e < PER; ++e) {
                        c[e] = tid * PER + e < entries ? sPre[tid * PER + e] : 0u;
                        sum += c[e];
                    }
                    uint32_t const incl = waveInclusiveScan(sum);
                    uint32_t acc = incl - sum;
#pragma unroll
                    for (int e = 0; e < PER; ++e) {
                        if (tid * PER + e < entries) sPre[tid * PER + e] = acc;
                        acc += c[e];
                    }
                    if (tid == 63) sPre[kPushMaxIters * kPushWaves] = incl;
                }
                __syncthreads();
                L = (int)sPre[kPushMaxIters * kPushWaves];
                if (a.stageShift && L <= kLeaverListLds) {
                    stageFromBits(S, sc, n, iters, bits, L, sPre, sGroup, sWaveCnt, sList);
                    continue;
                }
                for (int it = 0; it < iters; ++it) {
                    bool const left = (bits >> it) & 1u;
                    unsigned long long const m = __ballot(left);
                    if (left)
                        S.scratch[base + sPre[it * kPushWaves + wave] + (uint32_t)__popcll(m & laneMaskLt())] =
                            it * kPushThreads + tid;
                }
            } else {  // more particles than bits: the leavers from their multiMask
                for (int c0 = 0; c0 < n; c0 += kPushThreads) {
                    int const i = c0 + tid;
                    bool const left = i < n && S.mask[base + i] >= 2;
                    int total;
                    int const r = blockRank<kPushWaves>(left, sWaveCnt, &total);
                    if (left) S.scratch[base + L + r] = i;
                    L += total;
                }
            }
            __syncthreads();
            groupLeavers<kPushWaves>(S, sc, L, sGroup, sWaveCnt);
            if (a.stageShift) stageSC<kPushWaves>(S, sc, L, sWaveCnt);
        }
    }
}

// What bounds the kernel (TSC, Boris, 33.5M particles a launch): the LDS, whose
// bank conflicts follow from 64 lanes at unrelated cells, and the vector
// issue, both near 80 % of the launch. Before the aligned reads of the E/B
// tile and the one-word queue the LDS was busy 86 % of it and the vector
// units 73 %; on the 256^3 two-species shear flow a pass of five steps went
// from 150.1 to 126 ms.
// Waves per SIMD the register budget must allow. TSC and PQS: at most 128
// VGPRs, two workgroups per CU. TSC at 80 VGPRs has room for three, but the
// loop then spills (126 ms a pass against 133 to 142 with 80 VGPRs), and
// workgroups of 320 to 768 threads measured 12 to 28 % slower than 512. CIC
// needs 80 VGPRs, three workgroups.
template <int SUPP, int PUSHER, int MODE, bool EMZ = false>
__global__ __launch_bounds__(kPushThreads, SUPP == 2 ? 6 : 4) void kPushDeposit(PushArgs a) {
    __shared__ __align__(16) unsigned char smem[PushLds<SUPP, MODE>::BYTES];
    pushDepositSC<SUPP, PUSHER, MODE, EMZ>(a, a.scList[blockIdx.x], smem);
}

// the same with the PML's weight damping of absorbing species (a kernel of
// its own: the FP64 pow and exp of the damping would raise the register
// pressure of every launch)
template <int SUPP, int PUSHER, int MODE, bool EMZ = false>
__global__ __launch_bounds__(kPushThreads, SUPP == 2 ? 6 : 4) void kPushDepositPml(PushArgs a) {
    __shared__ __align__(16) unsigned char smem[PushLds<SUPP, MODE>::BYTES];
    pushDepositSC<SUPP, PUSHER, MODE, EMZ, true>(a, a.scList[blockIdx.x], smem);
}

// Batched form for ensembles: work items (simulation, supercell) of one
// checkerboard phase of every simulation in one launch; a workgroup takes
// items blockIdx.x, blockIdx.x + gridDim.x, ... so a grid smaller than the
// item count runs persistently. The member's arguments are read as constant
// memory (the table does not change while the kernel runs) at a uniform
// index, so they come by scalar loads as a kernel's own arguments do; as
// ordinary memory that stores might change they were held in vector
// registers (240 bytes per lane spilled, one workgroup less per CU). The loop
// over items still leaves 152 (CIC) to 300 bytes (PQS) per lane in scratch,
// where the plain kernel has none.
template <int SUPP, int PUSHER, int MODE, bool EMZ = false>
__global__ __launch_bounds__(kPushThreads, SUPP == 2 ? 6 : 4) void kPushDepositBatch(const PushArgs* __restrict__ table,
                                                                  const int2* __restrict__ work, int nwork) {
    __shared__ __align__(16) unsigned char smem[PushLds<SUPP, MODE>::BYTES];
    for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
        int2 const it = work[w];
        uintptr_t at = reinterpret_cast<uintptr_t>(table + __builtin_amdgcn_readfirstlane(it.x));
        asm volatile("" : "+s"(at));  // hides where the address comes from, so the cast below stays
        auto const entry = (const __attribute__((address_space(4))) PushArgs*)at;
        pushDepositSC<SUPP, PUSHER, MODE>(*(const PushArgs*)entry, __builtin_amdgcn_readfirstlane(it.y), smem);
        __syncthreads();  // the next item reuses the LDS
    }
}

hipError_t launchPushBatch(int supp, int pusher, const PushArgs* table, const int2* work, int nwork, int nblocks,
                           hipStream_t s) {
    if (nwork <= 0) return hipSuccess;
    if (nblocks <= 0 || nblocks > nwork) nblocks = nwork;
    switch (pusher * 8 + supp) {
#define PIC_BATCH_CASE(P, S)                                                                                        \
    case P * 8 + S:                                                                                                 \
        hipLaunchKernelGGL((kPushDepositBatch<S, P, 1>), dim3(nblocks), dim3(kPushThreads), 0, s, table, work, nwork); \
        break;
        PIC_BATCH_CASE(PIC_PUSHER_BORIS, 2)
        PIC_BATCH_CASE(PIC_PUSHER_BORIS, 3)
        PIC_BATCH_CASE(PIC_PUSHER_BORIS, 4)
        PIC_BATCH_CASE(PIC_PUSHER_VAY, 2)
        PIC_BATCH_CASE(PIC_PUSHER_VAY, 3)
        PIC_BATCH_CASE(PIC_PUSHER_VAY, 4)
        PIC_BATCH_CASE(PIC_PUSHER_HIGUERA_CARY, 2)
        PIC_BATCH_CASE(PIC_PUSHER_HIGUERA_CARY, 3)
        PIC_BATCH_CASE(PIC_PUSHER_HIGUERA_CARY, 4)
#undef PIC_BATCH_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int SUPP, int PUSHER, int MODE, bool EMZ>
static hipError_t launchT(const PushArgs& a, int nblocks, hipStream_t s) {
    if (MODE != 2 && a.damp.axes)
        hipLaunchKernelGGL((kPushDepositPml<SUPP, PUSHER, MODE, EMZ>), dim3(nblocks), dim3(kPushThreads), 0, s, a);
    else
        hipLaunchKernelGGL((kPushDeposit<SUPP, PUSHER, MODE, EMZ>), dim3(nblocks), dim3(kPushThreads), 0, s, a);
    return hipGetLastError();
}

template <int SUPP, bool EMZ>
static hipError_t launchS(int pusher, int mode, const PushArgs& a, int nblocks, hipStream_t s) {
    if (mode == 2) return launchT<SUPP, PIC_PUSHER_BORIS, 2, EMZ>(a, nblocks, s);
    if (mode == 0) {  // no deposit: the current solver does not matter
        if (pusher == PIC_PUSHER_VAY) return launchT<SUPP, PIC_PUSHER_VAY, 0, false>(a, nblocks, s);
        if (pusher == PIC_PUSHER_HIGUERA_CARY) return launchT<SUPP, PIC_PUSHER_HIGUERA_CARY, 0, false>(a, nblocks, s);
        return launchT<SUPP, PIC_PUSHER_BORIS, 0, false>(a, nblocks, s);
    }
    if (pusher == PIC_PUSHER_VAY) return launchT<SUPP, PIC_PUSHER_VAY, 1, EMZ>(a, nblocks, s);
    if (pusher == PIC_PUSHER_HIGUERA_CARY) return launchT<SUPP, PIC_PUSHER_HIGUERA_CARY, 1, EMZ>(a, nblocks, s);
    return launchT<SUPP, PIC_PUSHER_BORIS, 1, EMZ>(a, nblocks, s);
}

size_t pushTileElems(int supp) {
    switch (supp) {
        case 2: return PushLds<2, 1>::J_ELEMS;
        case 3: return PushLds<3, 1>::J_ELEMS;
        case 4: return PushLds<4, 1>::J_ELEMS;
        default: return 0;
    }
}

// One axis of a supercell's neighbourhood for the gather flush: the steps -1,
// 0, 1 to the supercells whose J tiles reach into it, in ascending
// checkerboard colour, and those supercells' indices (-1 beyond an open
// border). All values are uniform in the block.
struct CoverAxis {
    int step[3], sc[3];
};
__device__ __forceinline__ CoverAxis coverAxis(int s, int nsc, bool open, const uint8_t* __restrict__ colour) {
    CoverAxis a;
    int col[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {  // the supercell above first, as equal colours (rings of two) stay in order
        int t = s + 1 - k;
        bool const beyond = t < 0 || t >= nsc;
        t = t < 0 ? t + nsc : (t >= nsc ? t - nsc : t);
        a.step[k] = 1 - k;
        a.sc[k] = beyond && open ? -1 : t;
        col[k] = colour[t];
    }
#pragma unroll
    for (int pass = 0; pass < 3; ++pass) {  // (0,1), (1,2), (0,1)
        int const m = pass & 1;
        if (col[m] > col[m + 1]) {
            int const c = col[m], st = a.step[m], sc = a.sc[m];
            col[m] = col[m + 1], a.step[m] = a.step[m + 1], a.sc[m] = a.sc[m + 1];
            col[m + 1] = c, a.step[m + 1] = st, a.sc[m + 1] = sc;
        }
    }
    return a;
}

// pointers that come from a table in memory are generic to the compiler, and a
// flat load waits with the scalar and LDS operations: global memory stated
typedef const __attribute__((address_space(1))) float* GlobalFloats;

// Component C of one supercell's 256 J cells, a thread each: the values of
// the at most 2 x 2 x 3 tiles that cover a cell, all loaded before the first
// addition, then added as the flush adds them, in ascending checkerboard
// phase (zeros add nothing). A phase's index is colour_x + ncol_x (colour_y +
// ncol_y colour_z), so visiting z, then y, then x neighbours each in
// ascending colour is ascending phase (every supercell covering a cell lies
// in another phase). Bit k of `held` is 0 for a neighbour beyond an open
// border and for one whose tile is not written.
template <int SUPP, int C, bool BATCH>
__device__ __forceinline__ void gatherFlushComponent(const GridDev& g, const float* __restrict__ tiles,
                                                     const CoverAxis& ax, const CoverAxis& ay, const CoverAxis& az,
                                                     uint32_t held, float* __restrict__ J, size_t cell, bool fresh) {
    constexpr int DLO = Esirkepov<SUPP>::lowerMargin;
    using TG = JTileGeom<DLO, Esirkepov<SUPP>::upperMargin>;
    constexpr int J_ELEMS = PushLds<SUPP, 1>::J_ELEMS;
    constexpr int EX = TG::ext(C, 0), EY = TG::ext(C, 1), EZ = TG::ext(C, 2);
    int const tid = threadIdx.x;
    int const lx = tid & 7, ly = (tid >> 3) & 7, lz = tid >> 6;
    int const lane = (lz * EY + ly) * EX + lx;
    float w[27];
    // batched: opaque, so that the tiles' addresses are formed per component
    // (kept for all three they spilled 40 scalar registers; the plain kernel is
    // faster with them). 32 boxes of 32 to 96 cells an axis, five steps: 39.0
    // ms with them, 38.5 without, 38.3 before the tiles' words were read.
    int nscx = g.nscx;
    if (BATCH) asm volatile("" : "+s"(nscx));
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        int const a = k / 9, b = (k / 3) % 3, d = k % 3;
        int const ox = DLO - SCX * ax.step[d], oy = DLO - SCY * ay.step[b], oz = DLO - SCZ * az.step[a];
        w[k] = 0.0f;
        int const sc = ax.sc[d] + nscx * (ay.sc[b] + g.nscy * az.sc[a]);
        GlobalFloats const t = (GlobalFloats)tiles + (ptrdiff_t)sc * J_ELEMS + TG::off(C) + (oz * EY + oy) * EX + ox;
        // one predicate per load (no branch), so that the loads stay together
        bool const covers = ((unsigned)(lx + ox) < (unsigned)EX) & ((unsigned)(ly + oy) < (unsigned)EY) &
                            ((unsigned)(lz + oz) < (unsigned)EZ) & (((held >> k) & 1u) != 0u);
        if (covers) w[k] = t[lane];
    }
    auto const j = (__attribute__((address_space(1))) float*)J + cell;
    float v = fresh ? 0.0f : *j;
#pragma unroll
    for (int k = 0; k < 27; ++k) v += w[k];
    *j = v;
}

// J of one supercell (256 threads). fresh: J holds nothing yet (the sums
// start at zero and every cell is written), so the step needs no reset of J.
// 64^3 cells (CIC): 21 us a launch plus 5 for the reset with a loop of
// dependent loads over the candidates of every cell. The tiles of supercells
// without particles are neither written nor read: with zero tiles a nearly
// empty box of 192x128x160 cells (TSC, 15,360 supercells) took 0.40 ms a step
// in one launch and 0.28 by phases, now 0.25; a laser box of 96x512x64 cells,
// four fifths vacuum, 8.76 and 7.59 ms for ten steps.
template <int SUPP, bool BATCH>
__device__ __forceinline__ void gatherFlushSC(const GridDev& g, const float* __restrict__ tiles,
                                              const uint32_t* __restrict__ tileHeld,
                                              const uint8_t* __restrict__ colour, float* J0, float* J1, float* J2,
                                              int sc, bool fresh) {
    int const sx = sc % g.nscx, sy = (sc / g.nscx) % g.nscy, sz = sc / (g.nscx * g.nscy);
    CoverAxis const ax = coverAxis(sx, g.nscx, (g.open & 1) != 0, colour);
    CoverAxis const ay = coverAxis(sy, g.nscy, (g.open & 2) != 0, colour + g.nscx);
    CoverAxis const az = coverAxis(sz, g.nscz, (g.open & 4) != 0, colour + g.nscx + g.nscy);
    int const tid = threadIdx.x;
    uint32_t held;
    {  // lane k of each wave looks at neighbour k
        int const k = tid & 63, a = k / 9, b = (k / 3) % 3, d = k % 3;
        int const x = d == 0 ? ax.sc[0] : (d == 1 ? ax.sc[1] : ax.sc[2]);
        int const y = b == 0 ? ay.sc[0] : (b == 1 ? ay.sc[1] : ay.sc[2]);
        int const z = a == 0 ? az.sc[0] : (a == 1 ? az.sc[1] : az.sc[2]);
        bool const inBox = k < 27 && x >= 0 && y >= 0 && z >= 0;
        held = (uint32_t)__ballot(inBox && tileHeld[x + g.nscx * (y + g.nscy * z)] != 0u);
    }
    size_t const cell = (size_t)(sx * SCX + (tid & 7)) +
                        (size_t)g.nx * ((size_t)(sy * SCY + ((tid >> 3) & 7)) + (size_t)g.ny * (sz * SCZ + (tid >> 6)));
    gatherFlushComponent<SUPP, 0, BATCH>(g, tiles, ax, ay, az, held, J0, cell, fresh);
    if (BATCH) asm volatile("" : "+s"(held) : : "memory");
    gatherFlushComponent<SUPP, 1, BATCH>(g, tiles, ax, ay, az, held, J1, cell, fresh);
    if (BATCH) asm volatile("" : "+s"(held) : : "memory");
    gatherFlushComponent<SUPP, 2, BATCH>(g, tiles, ax, ay, az, held, J2, cell, fresh);
}

template <int SUPP>
__global__ __launch_bounds__(SCV) void kGatherFlush(GridDev g, const float* __restrict__ tiles,
                                                     const uint32_t* __restrict__ held,
                                                     const uint8_t* __restrict__ colour, float* J0, float* J1,
                                                     float* J2, int fresh) {
    if (halted(g)) return;
    gatherFlushSC<SUPP, false>(g, tiles, held, colour, J0, J1, J2, (int)blockIdx.x, fresh != 0);
}

template <int SUPP>
__global__ __launch_bounds__(SCV) void kGatherFlushBatch(const GatherEntry* __restrict__ table,
                                                          const int2* __restrict__ blocks, int fresh) {
    int2 const it = blocks[blockIdx.x];
    GatherEntry const e = table[__builtin_amdgcn_readfirstlane(it.x)];
    if (halted(e.g)) return;
    gatherFlushSC<SUPP, true>(e.g, e.tiles, e.held, e.colour, e.J[0], e.J[1], e.J[2], __builtin_amdgcn_readfirstlane(it.y),
                        fresh != 0);
}

hipError_t launchGatherFlushBatch(int supp, const GatherEntry* table, const int2* blocks, int nblocks, bool fresh,
                                  hipStream_t s) {
    if (nblocks <= 0) return hipSuccess;
    dim3 const grid(nblocks), block(SCV);
    switch (supp) {
        case 2: hipLaunchKernelGGL(kGatherFlushBatch<2>, grid, block, 0, s, table, blocks, fresh ? 1 : 0); break;
        case 3: hipLaunchKernelGGL(kGatherFlushBatch<3>, grid, block, 0, s, table, blocks, fresh ? 1 : 0); break;
        case 4: hipLaunchKernelGGL(kGatherFlushBatch<4>, grid, block, 0, s, table, blocks, fresh ? 1 : 0); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launchGatherFlush(int supp, const GridDev& g, const float* tiles, const uint32_t* held,
                             const uint8_t* colour, float* const J[3], bool fresh, hipStream_t s) {
    dim3 const grid((unsigned)(g.nscx * g.nscy * g.nscz)), block(SCV);
    int const f = fresh ? 1 : 0;
    switch (supp) {
        case 2: hipLaunchKernelGGL(kGatherFlush<2>, grid, block, 0, s, g, tiles, held, colour, J[0], J[1], J[2], f); break;
        case 3: hipLaunchKernelGGL(kGatherFlush<3>, grid, block, 0, s, g, tiles, held, colour, J[0], J[1], J[2], f); break;
        case 4: hipLaunchKernelGGL(kGatherFlush<4>, grid, block, 0, s, g, tiles, held, colour, J[0], J[1], J[2], f); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launchPush(int supp, int pusher, int mode, int currentSolver, const PushArgs& a, int nblocks,
                      hipStream_t s) {
    if (nblocks <= 0) return hipSuccess;
    bool const emz = currentSolver == PIC_CURRENT_SOLVER_EMZ;
    switch (supp) {
        case 2: return emz ? launchS<2, true>(pusher, mode, a, nblocks, s) : launchS<2, false>(pusher, mode, a, nblocks, s);
        case 3: return emz ? launchS<3, true>(pusher, mode, a, nblocks, s) : launchS<3, false>(pusher, mode, a, nblocks, s);
        case 4: return emz ? launchS<4, true>(pusher, mode, a, nblocks, s) : launchS<4, false>(pusher, mode, a, nblocks, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pic
