#pragma once
// tauhip_resident.h — the resident sweep: many half-sweeps of a volume that
// fits on the chip, in one launch.
//
// The streaming sweep (tauhip_sweep.h) pays, per launch of at most six
// half-sweeps, a launch, a pass over the field and the filling of its plane
// pipeline: 15 us for any volume up to 100^3, where the updates themselves
// take a tenth of that.  Here every workgroup keeps its tile of the volume in
// registers for the whole launch, so a half-sweep moves only tile faces, and
// no voxel is updated twice.  Per half-sweep, streaming and resident, on
// MI355X (256 compute units):
//   32^3 2.9, 1.2 us; 100^3 3.3, 1.5; 128^3 3.7, 1.7; 160^3 5.4, 3.2;
//   203 x 157 x 181 7.4, 4.3; 200^3 7.8, 4.6; 220^3 7.1, 5.8;
//   256^3 11.3, 6.2; 611 x 803 pixels 18, 1.8; 1500 x 1600 60, 2.5;
//   per-voxel field 128^3 6.4, 1.8, two of them 10, 2.9;
//   three-phase 128^3 5.5, 2.0, 160^3 8.0, 5.5; seven values
//   121 x 130 x 143 10.1, 4.4
// Bound: up to 128^3 the exchange of the faces (without it 0.4 to 0.8 us),
// beyond it issue and the exchange about evenly (200^3: 3.5 us without it).
//
// Mapping.  One axis of the volume (z, or y for a 2-D image, whose z is 1)
// lies along the lanes: lane l of a wave holds the P consecutive voxels from
// l * P of a row.  A wave owns a patch of PX x PY rows (x by the other axis),
// a workgroup WX x WY such patches.  x and row neighbours inside a patch are
// registers and the lane neighbour of a row's end voxels comes by DPP; the
// rows that other waves need go through LDS after each half-sweep (one
// barrier; two where the rows of both colours would not fit), those that
// other workgroups need through a mailbox in global memory.
//
// Mailbox.  A message is one 8-byte word, the voxel's value and a tag that
// counts half-sweeps across launches, written and read with relaxed
// device-scope atomics, so no flag, fence or second round trip follows the
// data: 1.0 to 1.3 us from the update of a border row to its use in another
// workgroup.  Two slots per row suffice: a wave sends half-sweep t + 1's rows after
// it has read its partner's of t, which the partner sent after reading the
// slot that is written again.
//
// Progress.  The workgroups wait for each other, so all of them have to be
// resident: the launch checks the grid against the occupancy.  Other work on
// the device can still hold compute units (another stream's resident sweep
// for ever), so every wait is bounded: a wave that has polled `spin` times
// records the launch in *status, stops waiting for the rest of the launch and
// still runs it to its end.  A launch that finds *status set returns at once
// and writes nothing; src is never written.  The caller reads the status
// with the sums of its next check and repeats the lost launches with the
// streaming sweep.

#include "tauhip_sweep.h"

struct ResidentArgs {
    const float* src;
    float* dst;
    const void* codes;     // as tf_sweep: sweep codes, face sections or face codes
    const float* table;    // as tf_sweep
    int n_table;           // face codes: its length
    long long fsec;        // field kind: floats between the face sections
    Vol v;
    int lane_n, row_n;  // extents of the lane axis and the row axis
    int sL, sR;         // their strides in the padded volume
    int cL, cR, cX;     // strides of the sweep codes: lane axis, row axis, x
    float w;
    int colour0, n_half;
    int WY, nTx, nTy, total;
    unsigned long long* mail;
    uint32_t tag0;
    int* status;
    int launch_id;
    int spin;
};

constexpr int kResidentSpin = 1 << 16;  // polls of one wait, about 50 ms

// (1/f, f) of a prefactor table entry for the reciprocal division of the
// anisotropic and electrode kinds; inf (an inert voxel) is the pair (0, 0).
// q = s (1/f) and one residual correction is s / f correctly rounded for a
// correctly rounded 1/f, f in [2^-20, 2^20] and |s| >= 2^-100 (Markstein's
// correction step: the residual is exact); `odd` reports a prefactor outside
// that range (a NaN among them), for which a launch divides throughout.
__device__ __forceinline__ void prefactor_pair(float f, float& r, float& g, bool& odd) {
    const bool inert = f == __builtin_inff();
    odd = !inert && !(f >= 0x1p-20f && f <= 0x1p20f);
    r = inert ? 0.0f : 1.0f / f;
    g = inert ? 0.0f : f;
}

template <int KIND>
constexpr int resident_table_floats() {
    return KIND == TF_KIND_SOLVER ? 18
           : KIND == TF_KIND_FIELD ? 0
           : KIND == TF_KIND_MULTIPHASE_FACES ? TF_RESIDENT_TABLE
           : 2 * (KIND == TF_KIND_ELECTRODE ? TF_ELECTRODE_TABLE : TF_ANISO_TABLE);
}

template <int KIND, int P, int PX, int PY, int NW>
struct ResidentShape {
    static constexpr int R = PX * PY;           // rows of a wave
    static constexpr int HP = P / 2;            // voxels of one colour per lane and row
    static constexpr int E = R * P;             // voxels per lane
    static constexpr int ROW = HP * 64;         // floats of one colour of a row
    static constexpr bool kEven = PX % 2 == 0 && PY % 2 == 0;
    static constexpr int inner(int p) { return p > 2 ? p - 2 : 0; }
    static constexpr int RB = R - inner(PX) * inner(PY);  // border rows of a patch
    static constexpr bool border(int row) {
        const int ix = row / PY, iy = row % PY;
        return ix == 0 || ix == PX - 1 || iy == 0 || iy == PY - 1;
    }
    // rows in the order of their update, the border rows first, and a border
    // row's place among them
    static constexpr int order(int n) {
        int seen = 0;
        for (int pass = 0; pass < 2; ++pass)
            for (int row = 0; row < R; ++row)
                if (border(row) == (pass == 0) && seen++ == n) return row;
        return 0;
    }
    static constexpr int place(int row) {
        int n = 0;
        for (int i = 0; i < row; ++i) n += border(i);
        return n;
    }
    // LDS in floats: the prefactor table, the published border rows of one
    // colour (two buffers where they fit), the tile's outer faces, and a
    // side of zeros
    // (the rows with ix = 0 come first and those with ix = PX - 1 last)
    static constexpr int PUB = NW * RB * ROW;
    static constexpr int ZERO = (PX > PY ? PX : PY) * ROW;
    static constexpr int HEAD = (resident_table_floats<KIND>() + 4 + 63) / 64 * 64;
    static constexpr int face(int wy) { return 2 * (wy * PY + NW / wy * PX) * ROW; }
    static constexpr int least_face() {
        int best = face(1);
        for (int wy = 2; wy <= NW; ++wy) best = NW % wy == 0 && face(wy) < best ? face(wy) : best;
        return best;
    }
    static constexpr int LDS = 160 * 256;  // floats of LDS in a compute unit
    static constexpr int NBUF = HEAD + 2 * PUB + least_face() + ZERO <= LDS ? 2 : 1;
    static constexpr size_t lds_floats(int wy) { return (size_t)HEAD + NBUF * PUB + face(wy) + ZERO; }
};

// Q0: the launch's first colour where the patch has even sides, else 0
template <int KIND, int P, int PX, int PY, int NW, bool PER, int Q0>
__global__ __launch_bounds__(NW * 64) void k_resident(ResidentArgs a) {
    using Sh = ResidentShape<KIND, P, PX, PY, NW>;
    constexpr int R = Sh::R, RB = Sh::RB, HP = Sh::HP, E = Sh::E, ROW = Sh::ROW, NBUF = Sh::NBUF, PUB = Sh::PUB;
    constexpr int NK = (E + 3) / 4;
    constexpr int kTable = resident_table_floats<KIND>();
    // per-voxel field: every face conductance in a register; MultiPhase face
    // codes: a code word per voxel; the others: a code byte per voxel
    constexpr bool kField = KIND == TF_KIND_FIELD, kFaceCodes = KIND == TF_KIND_MULTIPHASE_FACES;
    constexpr bool kBytes = !kField && !kFaceCodes;
    constexpr bool kPairs = KIND == TF_KIND_ANISOTROPIC || KIND == TF_KIND_ELECTRODE;
    static_assert(P % 2 == 0 && P >= 2, "a lane holds whole red/black pairs");

    // consecutive tiles on one XCD, as k_sweep
    const int per = gridDim.x >> 3;
    const int T = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (T >= a.total) return;

    extern __shared__ __align__(16) float rs_smem[];
    int* const s_flag = reinterpret_cast<int*>(rs_smem + kTable);  // [0] lost earlier, [1] prefactor out of range
    float* const pub = rs_smem + Sh::HEAD;
    float* const zero = pub + NBUF * PUB;
    float* const faces = zero + Sh::ZERO;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int WY = a.WY, WX = NW / WY;
    const int b = T / (a.nTx * a.nTy), tt = T - b * a.nTx * a.nTy;
    const int tx = tt / a.nTy, ty = tt - tx * a.nTy;
    const int NGX = (a.v.X + PX - 1) / PX, NGY = (a.row_n + PY - 1) / PY;
    const int wx = wave / WY, wy = wave - wx * WY;
    const int gx = tx * WX + wx, gy = ty * WY + wy;
    const bool live = gx < NGX && gy < NGY;

    if (threadIdx.x == 0) {
        s_flag[0] = __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_flag[1] = 0;
    }
    __syncthreads();
    if (s_flag[0] != 0) return;  // the same for the whole workgroup
    // zeros, also in the face rows: lanes past a row's end get no messages,
    // and what they hold must stay finite (their neighbours' DPP reads it)
    for (int i = threadIdx.x; i < Sh::ZERO + Sh::face(a.WY); i += NW * 64) zero[i] = 0.0f;
    if constexpr (KIND == TF_KIND_SOLVER) {
        if (threadIdx.x < kTable) rs_smem[threadIdx.x] = c_rd[threadIdx.x];
    } else if constexpr (kFaceCodes) {
        for (int i = threadIdx.x; i < a.n_table; i += NW * 64) rs_smem[i] = a.table[i];
    } else if constexpr (kPairs) {
        const float* tab = KIND == TF_KIND_ELECTRODE ? a.table + (size_t)b * TF_ELECTRODE_TABLE : a.table;
        for (int i = threadIdx.x; i < kTable / 2; i += NW * 64) {
            float r, f;
            bool odd;
            prefactor_pair(tab[i], r, f, odd);
            rs_smem[2 * i] = r;
            rs_smem[2 * i + 1] = f;
            if (odd) s_flag[1] = 1;
        }
    }

    // ---- the wave's patch ----
    // One descriptor per row, its record count 0 outside the volume, so that
    // those rows and the lanes past the row's end read zeros.  What lies
    // between the row's last voxel and the end of its last lane's elements
    // has code 0, so its value stays 0 whatever its neighbours hold.
    const float* const S = a.src + (size_t)b * a.v.sB;
    const int l0 = lane * P;
    // the lane's P words of the row whose first voxel is word o of `base`
    auto load_row = [&](const float* base, size_t o, bool ok, float (&d)[P]) {
        const rsrc_t r = make_rsrc(base + (ok ? o : 0), ok ? (uint32_t)((a.lane_n - 1) * a.sL + 1) * 4u : 0u);
        const int vo = l0 * a.sL * 4;
        if (a.sL == 1 && P == 2) {
            const u32x2_t q = __builtin_amdgcn_raw_buffer_load_b64(r, vo, 0, 0);
            d[0] = lo_f(q);
            d[1] = hi_f(q);
        } else if (a.sL == 1) {
            typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int e = 0; e + 3 < P; e += 4) {
                const u32x4_t q = __builtin_amdgcn_raw_buffer_load_b128(r, vo + 4 * e, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t u = q[i];
                    d[e + i] = __builtin_bit_cast(float, u);
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < P; ++e) d[e] = ld_f32(r, vo, e * a.sL * 4);
        }
    };
    // word of voxel (x, r) of the patch's plane and row, the lane axis's first
    auto word_at = [&](int x, int r) {
        return (size_t)(x + 1) * a.v.sX + (size_t)(r + 1) * a.sR + a.sL;
    };
    float F[R][P];
    uint32_t K[kBytes ? NK : 1];
#pragma unroll
    for (int i = 0; i < (kBytes ? NK : 1); ++i) K[i] = 0;
    // the words of the voxels and of their neighbours on the minus sides,
    // which hold those faces (lane axis: of the row's element before the
    // lane's first)
    constexpr int NS = kField ? 3 : kFaceCodes ? 1 : 0;  // words per voxel: x, row, lane faces
    float G[NS > 0 ? NS : 1][R][P], Gx[PY][P], Gr[PX][P], Gl[R];
    float wrow[PX];           // 0 in rows past the volume: a ghost row keeps its value
    float first, last[PX];    // 1 in the first and the last layer (their x faces count twice)
    const float* const W = kBytes ? S : reinterpret_cast<const float*>(a.codes) + (size_t)b * a.v.sB;
    const float* const Wr = W + (kField ? (a.sL == 1 ? 1 : 2) * a.fsec : 0);  // row-axis faces
    const float* const Wl = W + (kField ? (a.sL == 1 ? 2 : 1) * a.fsec : 0);  // lane-axis faces
    first = gx == 0 ? 1.0f : 0.0f;
#pragma unroll
    for (int ix = 0; ix < PX; ++ix) {
        const int x = gx * PX + ix;
        wrow[ix] = x < a.v.X ? a.w : 0.0f;
        last[ix] = x == a.v.X - 1 ? 1.0f : 0.0f;
#pragma unroll
        for (int iy = 0; iy < PY; ++iy) {
            const int r = gy * PY + iy, row = ix * PY + iy;
            const bool ok = live && x <= a.v.X && r < a.row_n, in = ok && x < a.v.X;
            load_row(S, word_at(x, r), ok, F[row]);
            if constexpr (NS > 0) {
                load_row(W, word_at(x, r), in, G[0][row]);
                if constexpr (kField) {
                    load_row(Wr, word_at(x, r), in, G[1][row]);
                    load_row(Wl, word_at(x, r), in, G[2][row]);
                }
                const size_t o = in ? word_at(x, r) - a.sL : 0;
                Gl[row] = ld_f32(make_rsrc(Wl + o, in ? (uint32_t)((a.lane_n - 1) * a.sL + 1) * 4u : 0u), l0 * a.sL * 4);
                if (ix == 0) load_row(W, word_at(x - 1, r), in, Gx[iy]);
                if (iy == 0) load_row(Wr, word_at(x, r - 1), in, Gr[ix]);
            } else {
                const uint8_t* const C =
                    reinterpret_cast<const uint8_t*>(a.codes) + (size_t)b * sweep_code_volume(a.v.X, a.v.Y, a.v.Z);
                // byte z + 3 of a code row is voxel z, the lane axis's first
                // voxel z = 1 (codes along z: up to the end of the row's last
                // word, zeros past Z)
                const size_t oc = in ? (size_t)(x + 1) * a.cX + (size_t)(r + 1) * a.cR + (a.cL == 1 ? 4 : a.cL + 3) : 0;
                const uint32_t nc = a.cL == 1 ? (uint32_t)a.cR - 4u : (uint32_t)((a.lane_n - 1) * a.cL + 1);
                const rsrc_t rC = make_rsrc(C + oc, in ? nc : 0u);
                const int vc = l0 * a.cL;
                if (a.cL == 1 && P == 2) {
                    K[row / 2] |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rC, vc, 0, 0) << (16 * (row % 2));
                } else if (a.cL == 1) {
#pragma unroll
                    for (int e = 0; e + 3 < P; e += 4)
                        K[(row * P + e) / 4] = __builtin_amdgcn_raw_buffer_load_b32(rC, vc + e, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < P; ++e)
                        K[(row * P + e) / 4] |= ld_u8(rC, vc, e * a.cL) << (8 * ((row * P + e) % 4));
                }
            }
        }
    }

    // ---- where each side's rows come from ----
    enum { kZero, kLds, kMail, kGhost };
    int sxm = kZero, sxp = kZero, srm = kZero, srp = kZero;
    int wxm = wave, wxp = wave, wrm = wave, wrp = wave;  // waves of the LDS sides
    int Txm = T, Txp = T, Trm = T, Trp = T;              // tiles of the mail sides
    if (live) {
        if (gx == 0) sxm = kGhost;
        else if (wx > 0) { sxm = kLds; wxm = wave - WY; }
        else { sxm = kMail; Txm = T - a.nTy; }
        if (gx == NGX - 1) sxp = (gx + 1) * PX == a.v.X ? kGhost : kZero;
        else if (wx < WX - 1) { sxp = kLds; wxp = wave + WY; }
        else { sxp = kMail; Txp = T + a.nTy; }
        auto row_side = [&](int g, int& s, int& w, int& t) {
            if (g < 0 || g >= NGY) {
                if (!PER) return;
                g = g < 0 ? NGY - 1 : 0;
            }
            const int ot = g / WY;
            if (ot == ty) { s = kLds; w = wx * WY + (g - ot * WY); }
            else { s = kMail; t = T + (ot - ty); }
        };
        row_side(gy - 1, srm, wrm, Trm);
        row_side(gy + 1, srp, wrp, Trp);
    }
    const int RYt = WY * PY, RXt = WX * PX, tile_rows = 2 * (RYt + RXt);
    typedef unsigned long long word_t;
    // mailbox places in bytes (the plan keeps it below 2 GiB): a row's words
    // of slot 0; the other slot is `slot` bytes on
    const uint32_t slot = (uint32_t)tile_rows * (ROW * 8);
    // place of a row among a tile's face rows: sides x-, x+, row-, row+
    auto face_row = [&](int side, int row) {
        return (side == 0 ? 0 : side == 1 ? RYt : side == 2 ? 2 * RYt : 2 * RYt + RXt) + row;
    };
    auto box = [&](int tile, int side, int row) {
        return (uint32_t)tile * (2 * slot) + (uint32_t)face_row(side, row) * (ROW * 8);
    };
    const uint32_t in_x = box(T, sxm == kMail ? 0 : 1, wy * PY);
    const uint32_t in_r = box(T, srm == kMail ? 2 : 3, wx * PX);
    const uint32_t out_xm = box(Txm, 1, wy * PY), out_xp = box(Txp, 0, wy * PY);
    const uint32_t out_rm = box(Trm, 3, wx * PX), out_rp = box(Trp, 2, wx * PX);
    // word i of this lane from a place
    // (from `at`, this lane's 8 bytes of a row, made anew where it is used:
    // otherwise every place keeps a register of its own through the loop)
    auto lane_bytes = [&]() {
        uint32_t v = (uint32_t)lane * 8u;
        asm volatile("" : "+v"(v));
        return v;
    };
    auto word_of = [&](uint32_t place, uint32_t at, int i) {
        return reinterpret_cast<word_t*>(reinterpret_cast<char*>(a.mail) + (place + at)) + i * 64;
    };
    // where the rows of a side that no wave of this workgroup publishes are kept
    float* const f_xm = faces + face_row(0, wy * PY) * ROW + lane;
    float* const f_xp = faces + face_row(1, wy * PY) * ROW + lane;
    float* const f_rm = faces + face_row(2, wx * PX) * ROW + lane;
    float* const f_rp = faces + face_row(3, wx * PX) * ROW + lane;
    const bool in_row = l0 < a.lane_n;  // the other lanes' words are not sent
    const bool mail_x = sxm == kMail || sxp == kMail, mail_r = srm == kMail || srp == kMail;
    // lane of the row's last voxel (periodic rows fill it: lane_n % P == 0)
    const int last_lane = PER ? a.lane_n / P - 1 : 0;

    // colour of the patch's first voxel: element e of row (ix, iy) is updated
    // in half-sweep t when e = Q ^ ix ^ iy (mod 2), Q = q0 ^ t (mod 2)
    const int q0 = Sh::kEven ? Q0 : (a.colour0 ^ (gx * PX) ^ (gy * PY)) & 1;
    bool dead = false;
    __syncthreads();
    const int rare_below = kPairs && s_flag[1] != 0 ? 1024 : -99;

    auto publish = [&](auto q_c, int buf) {
        constexpr int Q = decltype(q_c)::value;
        float* const p = pub + buf * PUB + wave * (RB * ROW) + lane;
        static_for<0, R>([&](auto r_c) {
            constexpr int row = decltype(r_c)::value, ae = (Q ^ (row / PY) ^ (row % PY)) & 1;
            if constexpr (Sh::border(row)) {
#pragma unroll
                for (int k = 0; k < HP; ++k) p[Sh::place(row) * ROW + k * 64] = F[row][2 * k + ae];
            }
        });
    };
    // the rows of the tile faces, tagged, into the other tiles' slot
    auto send = [&](auto q_c, uint32_t tag, int sl) {
        constexpr int Q = decltype(q_c)::value;
        const uint32_t lane8 = lane_bytes();
        auto put = [&](uint32_t place, int ix, int iy, int at) {
            const int row = ix * PY + iy, ae = (Q ^ ix ^ iy) & 1;
#pragma unroll
            for (int k = 0; k < HP; ++k) {
                // a copy: F itself would be allocated as half of the word
                float val = F[row][2 * k + ae];
                asm volatile("" : "+v"(val));
                __hip_atomic_store(word_of(place + sl * slot, lane8, at * HP + k),
                                   (word_t)tag << 32 | __builtin_bit_cast(uint32_t, val), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        if (!in_row) return;
        if (sxm == kMail)
#pragma unroll
            for (int iy = 0; iy < PY; ++iy) put(out_xm, 0, iy, iy);
        if (sxp == kMail)
#pragma unroll
            for (int iy = 0; iy < PY; ++iy) put(out_xp, PX - 1, iy, iy);
        if (srm == kMail)
#pragma unroll
            for (int ix = 0; ix < PX; ++ix) put(out_rm, ix, 0, ix);
        if (srp == kMail)
#pragma unroll
            for (int ix = 0; ix < PX; ++ix) put(out_rp, ix, PY - 1, ix);
    };

    const float ky = KIND == TF_KIND_ANISOTROPIC ? a.table[TF_ANISO_TABLE - 2] : 0.0f;
    const float kz = KIND == TF_KIND_ANISOTROPIC ? a.table[TF_ANISO_TABLE - 1] : 0.0f;
    // weights of the row axis and of the lane axis
    const float k_row = a.sL == 1 ? ky : kz, k_lane = a.sL == 1 ? kz : ky;
    // face codes: bits of the row axis's and of the lane axis's face
    const int sh_row = a.sL == 1 ? 6 : 12, sh_lane = a.sL == 1 ? 12 : 6;

    auto half = [&](auto q_c, int t) {
        constexpr int Q = decltype(q_c)::value;
        // the packed codes as if new in every half-sweep: the compiler would
        // otherwise keep every extracted byte in a register of its own
        // (the field kind: the sums of the faces, where they would not fit)
        if constexpr (kBytes) {
#pragma unroll
            for (int i = 0; i < NK; ++i) asm volatile("" : "+v"(K[i]));
        } else if constexpr (kFaceCodes || E > 8) {
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int e = 0; e < P; ++e) asm volatile("" : "+v"(G[0][i][e]));
        }
        // the x ghost plane xg next to row ix of the patch: constant
        auto ghost_x = [&](float* d, int xg, int ix) {
            const rsrc_t r = make_rsrc(S + (size_t)xg * a.v.sX, (uint32_t)a.v.sX * 4u);
#pragma unroll
            for (int iy = 0; iy < PY; ++iy) {
                const int ae = (Q ^ ix ^ iy) & 1;
#pragma unroll
                for (int k = 0; k < HP; ++k)
                    d[iy * ROW + k * 64] =
                        ld_f32(r, l0 * a.sL * 4, ((gy * PY + iy + 1) * a.sR + (1 + 2 * k + ae) * a.sL) * 4);
            }
        };
        if (sxm == kGhost) ghost_x(f_xm, 0, 0);
        if (sxp == kGhost) ghost_x(f_xp, a.v.X + 1, PX - 1);
        // a wave has at most one mail side per axis (the plan sees to it);
        // the words of both are asked for together
        auto poll = [&](auto hx_c, auto hr_c) {
            constexpr bool HX = decltype(hx_c)::value, HR = decltype(hr_c)::value;
            constexpr int NX = HX ? PY * HP : 0, N = NX + (HR ? PX * HP : 0);
            if (!in_row) return;
            const uint32_t tag = a.tag0 + (uint32_t)t;
            const uint32_t so = (t & 1) * slot, lane8 = lane_bytes();
            word_t m[N];
            for (int n = dead ? a.spin : 0;; ++n) {
                // (no pause, and one question at a time: a first question 0.3
                // us later, or two and three of them in flight 0.2 us apart,
                // cost 0.1 to 0.3 us per half-sweep from 32^3 to 200^3)
                bool ok = true;
#pragma unroll
                for (int i = 0; i < N; ++i)
                    m[i] = __hip_atomic_load(i < NX ? word_of(in_x + so, lane8, i) : word_of(in_r + so, lane8, i - NX),
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int i = 0; i < N; ++i) ok = ok && (uint32_t)(m[i] >> 32) == tag;
                if (__builtin_amdgcn_ballot_w64(!ok) == 0) break;
                if (n >= a.spin) {
                    if (!dead && lane == 0) atomicCAS(a.status, 0, a.launch_id);
                    dead = true;
                    break;
                }
            }
            float* const dx = sxm == kMail ? f_xm : f_xp;
            float* const dr = srm == kMail ? f_rm : f_rp;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float val = __builtin_bit_cast(float, (uint32_t)m[i]);
                if (i < NX) dx[i * 64] = val;
                else dr[(i - NX) * 64] = val;
            }
        };
        if (mail_x && mail_r) poll(std::true_type{}, std::true_type{});
        else if (mail_x) poll(std::true_type{}, std::false_type{});
        else if (mail_r) poll(std::false_type{}, std::true_type{});

        // a side's row lies in another wave's published rows, among the tile's
        // outer faces or in the zeros
        const float* const pb = pub + (NBUF == 2 ? (t + 1) & 1 : 0) * PUB + lane;
        const float* const e_xm = sxm == kLds ? pb + (wxm * RB + RB - PY) * ROW : sxm == kZero ? zero + lane : f_xm;
        const float* const e_xp = sxp == kLds ? pb + wxp * (RB * ROW) : sxp == kZero ? zero + lane : f_xp;
        const float* const e_rm = srm == kLds ? pb + wrm * (RB * ROW) : srm == kZero ? zero + lane : f_rm;
        const float* const e_rp = srp == kLds ? pb + wrp * (RB * ROW) : srp == kZero ? zero + lane : f_rp;
        // voxels I0 .. I0 + N - 1 of one colour, in the order of Sh::order:
        // every load first, one test for rare quotients
        auto update = [&](auto i_c, auto n_c) {
            constexpr int I0 = decltype(i_c)::value, N = decltype(n_c)::value;
            float s[N], q[N], f[N];
            bool rare = false;
            static_for<0, N>([&](auto j_c) {
                constexpr int j = decltype(j_c)::value, row = Sh::order((I0 + j) / HP), k = (I0 + j) % HP;
                constexpr int ix = row / PY, iy = row % PY, e = 2 * k + ((Q ^ ix ^ iy) & 1);
                float xm, xp, rm, rp, lm, lp;
                if constexpr (ix > 0) xm = F[row - PY][e]; else xm = e_xm[iy * ROW + k * 64];
                if constexpr (ix < PX - 1) xp = F[row + PY][e]; else xp = e_xp[iy * ROW + k * 64];
                if constexpr (iy > 0) rm = F[row - 1][e]; else rm = e_rm[(srm == kLds ? Sh::place(ix * PY + PY - 1) : ix) * ROW + k * 64];
                if constexpr (iy < PY - 1) rp = F[row + 1][e]; else rp = e_rp[(srp == kLds ? Sh::place(ix * PY) : ix) * ROW + k * 64];
                if constexpr (e > 0) {
                    lm = F[row][e - 1];
                } else {
                    const uint32_t end = __builtin_bit_cast(uint32_t, F[row][P - 1]);
                    if constexpr (PER) {
                        // lane 0 takes the row's last voxel
                        const int wrapped = __builtin_amdgcn_readlane((int)end, last_lane);
                        lm = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(wrapped, (int)end, 0x138, 0xf, 0xf, false));
                    } else {
                        lm = from_prev_lane(end);
                    }
                }
                if constexpr (e < P - 1) {
                    lp = F[row][e + 1];
                } else {
                    const uint32_t first = __builtin_bit_cast(uint32_t, F[row][0]);
                    lp = from_next_lane(first);
                    if constexpr (PER) {
                        const float wrapped = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane((int)first));
                        lp = lane == last_lane ? wrapped : lp;
                    }
                }
                if constexpr (kBytes) {
                    constexpr int at = row * P + e;
                    const uint32_t code = (K[at / 4] >> (8 * (at % 4))) & 0xffu;
                    const float2 rf = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(rs_smem) +
                                                                       (kPairs ? code * 8 : code));
                    float sum = xp + xm;
                    if constexpr (KIND == TF_KIND_ANISOTROPIC) {
                        float u = rp + rm;
                        u = k_row * u;
                        sum = sum + u;
                        u = lp + lm;
                        u = k_lane * u;
                        sum = sum + u;
                    } else {
                        sum = sum + rp;
                        sum = sum + rm;
                        sum = sum + lp;
                        sum = sum + lm;
                    }
                    s[j] = sum;
                    f[j] = rf.y;
                    q[j] = sum * rf.x;
                    const float res = __builtin_fmaf(-q[j], rf.y, sum);
                    q[j] = __builtin_fmaf(res, rf.x, q[j]);
                    // the reciprocal is not exact: a subnormal residual
                    // (Solver), a tiny sum, or nothing finite (prefactor_pair)
                    rare = rare || (kPairs ? __builtin_amdgcn_frexp_expf(sum) < rare_below ||
                                                 __builtin_amdgcn_classf(res, 0x207)
                                           : __builtin_amdgcn_classf(res, 0x90));
                } else {
                    // the six faces: the voxel's own plus faces and those of
                    // its neighbours on the minus sides
                    auto word = [](float w) { return __builtin_bit_cast(uint32_t, w); };
                    float wxm, wrm, wlm;
                    if constexpr (ix > 0) wxm = G[0][row - PY][e]; else wxm = Gx[iy][e];
                    if constexpr (iy > 0) wrm = G[kField ? 1 : 0][row - 1][e]; else wrm = Gr[ix][e];
                    if constexpr (e > 0) wlm = G[kField ? 2 : 0][row][e - 1]; else wlm = Gl[row];
                    float gxp, gxm, grp, grm, glp, glm;
                    if constexpr (kField) {
                        gxp = G[0][row][e], grp = G[1][row][e], glp = G[2][row][e];
                        gxm = wxm, grm = wrm, glm = wlm;
                    } else {
                        const char* const tb = reinterpret_cast<const char*>(rs_smem);
                        auto face = [tb](uint32_t c, int at) {
                            return *reinterpret_cast<const float*>(tb + ((c >> at) & 63u));
                        };
                        const uint32_t own = word(G[0][row][e]);
                        gxp = face(own, 0), grp = face(own, sh_row), glp = face(own, sh_lane);
                        gxm = face(word(wxm), 0), grm = face(word(wrm), sh_row), glm = face(word(wlm), sh_lane);
                    }
                    float sum = xp * gxp + xm * gxm;
                    sum = sum + rp * grp;
                    sum = sum + rm * grm;
                    sum = sum + lp * glp;
                    sum = sum + lm * glm;
                    if constexpr (kField) {
                        float fs = gxm + gxp;
                        fs = fs + grm;
                        fs = fs + grp;
                        fs = fs + glm;
                        fs = fs + glp;
                        // fma with a factor 0 or 1 rounds as the sum
                        if constexpr (ix == 0) fs = __builtin_fmaf(gxm, first, fs);
                        fs = __builtin_fmaf(gxp, last[ix], fs);
                        if (fs == 0.0f) fs = __builtin_inff();
                        q[j] = sum / fs;
                    } else {
                        const float2 rf = *reinterpret_cast<const float2*>(
                            reinterpret_cast<const char*>(rs_smem) + 4 * TF_MPF_FACE_SLOTS + (word(G[0][row][e]) >> 18));
                        s[j] = sum;
                        f[j] = rf.y;
                        q[j] = sum * rf.x;
                        const float res = __builtin_fmaf(-q[j], rf.y, sum);
                        q[j] = __builtin_fmaf(res, rf.x, q[j]);
                        rare = rare || __builtin_amdgcn_frexp_expf(sum) < -99;  // as rsweep_tile
                    }
                }
            });
            // those quotients are divided; the pair (0, 0) stands for an
            // infinite prefactor
            if (!kField && __builtin_expect(__builtin_amdgcn_ballot_w64(rare) != 0, 0)) {
#pragma unroll
                for (int j = 0; j < N; ++j) q[j] = f[j] != 0.0f ? s[j] / f[j] : s[j] / __builtin_inff();
            }
            static_for<0, N>([&](auto j_c) {
                constexpr int j = decltype(j_c)::value, row = Sh::order((I0 + j) / HP), k = (I0 + j) % HP;
                constexpr int ix = row / PY, iy = row % PY, e = 2 * k + ((Q ^ ix ^ iy) & 1);
                const float c = F[row][e];
                float d = q[j] - c;
                d = d * wrow[ix];
                F[row][e] = c + d;
            });
            if constexpr (kField) __builtin_amdgcn_sched_barrier(0);
        };
        auto update_all = [&](auto from_c, auto to_c) {
            constexpr int from = decltype(from_c)::value, to = decltype(to_c)::value;
            constexpr int M = kFaceCodes || (kField && E > 32) ? 2 : !kBytes || E <= 32 || E > 64 ? 4 : 8;  // quotients per test
            static_for<0, (to - from + M - 1) / M>([&](auto g_c) {
                constexpr int i = from + decltype(g_c)::value * M;
                update(ic<i>{}, ic<(to - i < M ? to - i : M)>{});
            });
        };
        // the border rows first: their messages are on the way while the
        // inner rows are updated
        update_all(ic<0>{}, ic<RB * HP>{});
        if (t + 1 < a.n_half) send(q_c, a.tag0 + (uint32_t)t + 1u, (t + 1) & 1);
        update_all(ic<RB * HP>{}, ic<R * HP>{});
    };

    // the voxels half-sweep 0 reads: those of the other colour
    if (live) {
        if (q0) {
            publish(ic<0>{}, NBUF == 2 ? 1 : 0);
            send(ic<0>{}, a.tag0, 0);
        } else {
            publish(ic<1>{}, NBUF == 2 ? 1 : 0);
            send(ic<1>{}, a.tag0, 0);
        }
    }
    __syncthreads();
    // one half-sweep and what it publishes; the barriers are the workgroup's
    auto step = [&](auto q_c, int t) {
        if (live) half(q_c, t);
        if constexpr (NBUF == 1) __syncthreads();  // the edges have been read
        if (live) publish(q_c, NBUF == 2 ? t & 1 : 0);
        __syncthreads();
    };
    if constexpr (Sh::kEven) {
        // every patch starts on the same colour, the kernel's own Q0: the two
        // colours' half-sweeps in a row, without a branch whose sides would
        // join the whole patch in other registers (128 voxels per lane: 74
        // registers spilled with it, none without)
        for (int t = 0; t < a.n_half; t += 2) {
            step(ic<Q0>{}, t);
            if (t + 1 == a.n_half) break;
            step(ic<Q0 ^ 1>{}, t + 1);
        }
    } else {
        // the patches differ in their first colour: a branch per wave, the
        // barriers outside of it
        for (int t = 0; t < a.n_half; ++t) {
            const bool odd = ((q0 ^ t) & 1) != 0;
            if constexpr (NBUF == 2) {
                if (live) {
                    if (odd) {
                        half(ic<1>{}, t);
                        publish(ic<1>{}, t & 1);
                    } else {
                        half(ic<0>{}, t);
                        publish(ic<0>{}, t & 1);
                    }
                }
            } else {
                if (live) {
                    if (odd) half(ic<1>{}, t);
                    else half(ic<0>{}, t);
                }
                __syncthreads();  // the edges have been read
                if (live) {
                    if (odd) publish(ic<1>{}, 0);
                    else publish(ic<0>{}, 0);
                }
            }
            __syncthreads();
        }
    }

    if (!live) return;
    float* const D = a.dst + (size_t)b * a.v.sB;
#pragma unroll
    for (int ix = 0; ix < PX; ++ix)
#pragma unroll
        for (int iy = 0; iy < PY; ++iy) {
            const int x = gx * PX + ix, r = gy * PY + iy, row = ix * PY + iy;
            if (x >= a.v.X || r >= a.row_n || l0 >= a.lane_n) continue;
            float* const d = D + (size_t)(x + 1) * a.v.sX + (size_t)(r + 1) * a.sR + (size_t)(l0 + 1) * a.sL;
            if (a.sL == 1 && l0 + P <= a.lane_n) {
                __builtin_memcpy(d, F[row], sizeof(F[row]));
            } else {
#pragma unroll
                for (int e = 0; e < P; ++e)
                    if (l0 + e < a.lane_n) d[(size_t)e * a.sL] = F[row][e];
            }
        }
}

template <int KIND, int P, int PX, int PY, int NW, bool PER, int Q0>
static int launch_resident_colour(const ResidentArgs& a, hipStream_t st) {
    using Sh = ResidentShape<KIND, P, PX, PY, NW>;
    const auto fn = k_resident<KIND, P, PX, PY, NW, PER, Q0>;
    const size_t lds = Sh::lds_floats(a.WY) * sizeof(float);
    if (lds > 160 * 1024) return fail(TF_NOT_RESIDENT, "a resident tile needs %zu B of LDS", lds);
    static bool attr_set = false;
    if (!attr_set) {
        if (hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
            (void)hipGetLastError();
        attr_set = true;
    }
    const int grid = (a.total + 7) / 8 * 8;
    // workgroups wait for each other: never launch more than are resident
    static int slots_cache[NW + 1][kMaxDevices] = {};  // per wy
    const int slots = resident_workgroups((const void*)fn, NW * 64, lds, slots_cache[a.WY]);
    if (grid > slots)
        return fail(TF_NOT_RESIDENT, "%d workgroups of the resident sweep exceed the %d resident ones", grid, slots);
    hipLaunchKernelGGL(fn, dim3(grid), dim3(NW * 64), lds, st, a);
    TF_LAUNCH_CHECK("k_resident");
    return 0;
}

template <int KIND, int P, int PX, int PY, int NW, bool PER>
static int launch_resident(const ResidentArgs& a, hipStream_t st) {
    if constexpr (ResidentShape<KIND, P, PX, PY, NW>::kEven)
        if (a.colour0) return launch_resident_colour<KIND, P, PX, PY, NW, PER, 1>(a, st);
    return launch_resident_colour<KIND, P, PX, PY, NW, PER, 0>(a, st);
}

// The compiled shapes, those that some volume's plan takes: (voxels per lane
// and row, patch rows in x, patch rows of the other axis, waves).  Up to 32
// voxels per lane the workgroup has 16 waves (128 registers per lane); larger
// patches need 8 (256 registers).  A spilled register's reload waits for
// every store before it, so one between the sends waits a microsecond for
// their acknowledgement.  That bounds each kind's patches; four kernels spill
// (face codes 8, 2, 4 15 registers in either colour and 8, 2, 3 2, field
// 4, 3, 3 8).
#define TF_RESIDENT_SHAPES_PAIRS(F) \
    F(2, 1, 1, 16) F(2, 1, 2, 16) F(2, 2, 2, 16) F(2, 2, 4, 16) F(2, 4, 4, 16) F(2, 6, 8, 8) \
    F(4, 1, 1, 16) F(4, 1, 2, 16) F(4, 2, 2, 16) F(4, 2, 3, 16) F(4, 2, 4, 16) F(4, 4, 6, 8) \
    F(8, 1, 1, 16) F(8, 1, 2, 16) F(8, 2, 2, 16) F(8, 2, 3, 8) F(8, 3, 4, 8) \
    F(16, 1, 1, 16) F(16, 2, 2, 8) F(32, 1, 1, 8)

// the Solver kind: 128 voxels per lane as well
#define TF_RESIDENT_SHAPES(F) TF_RESIDENT_SHAPES_PAIRS(F) F(2, 8, 8, 8) F(4, 4, 8, 8)

// Face codes take a word per voxel: half the voxels per register.
#define TF_RESIDENT_SHAPES_FACES(F) \
    F(2, 1, 1, 16) F(2, 1, 2, 16) F(2, 2, 2, 16) F(2, 2, 4, 16) F(2, 4, 6, 8) F(2, 4, 8, 8) \
    F(4, 1, 1, 16) F(4, 1, 2, 16) F(4, 2, 2, 16) F(4, 3, 3, 8) F(4, 2, 6, 8) F(4, 4, 4, 8) \
    F(8, 1, 1, 16) F(8, 1, 2, 16) F(8, 2, 3, 8) F(8, 2, 4, 8) F(16, 1, 1, 8) F(16, 1, 2, 8)

// The field kind takes three words per voxel.
#define TF_RESIDENT_SHAPES_FIELD(F) \
    F(2, 1, 1, 16) F(2, 1, 2, 16) F(2, 2, 2, 16) F(2, 2, 3, 16) F(2, 4, 4, 8) \
    F(4, 1, 1, 16) F(4, 1, 2, 16) F(4, 1, 3, 16) F(4, 2, 4, 8) F(4, 3, 3, 8) \
    F(8, 1, 1, 16) F(8, 1, 3, 8) F(8, 2, 2, 8) F(16, 1, 1, 8)

template <int KIND, bool PER>
static int dispatch_resident(const tf_resident& p, const ResidentArgs& a, hipStream_t st) {
#define F(P, PX, PY, NW) \
    if (p.elems == P && p.px == PX && p.py == PY && p.waves == NW) return launch_resident<KIND, P, PX, PY, NW, PER>(a, st);
    if constexpr (KIND == TF_KIND_FIELD) {
        TF_RESIDENT_SHAPES_FIELD(F)
    } else if constexpr (KIND == TF_KIND_MULTIPHASE_FACES) {
        TF_RESIDENT_SHAPES_FACES(F)
    } else if constexpr (KIND == TF_KIND_SOLVER) {
        TF_RESIDENT_SHAPES(F)
    } else {
        TF_RESIDENT_SHAPES_PAIRS(F)
    }
#undef F
    return fail(-1, "resident shape (%d, %d, %d, %d) is not compiled", p.elems, p.px, p.py, p.waves);
}

// per-kind entry points (one translation unit each)
int resident_dispatch_solver(const tf_resident& p, const ResidentArgs& a, hipStream_t st);
int resident_dispatch_periodic(const tf_resident& p, const ResidentArgs& a, hipStream_t st);
int resident_dispatch_anisotropic(const tf_resident& p, const ResidentArgs& a, hipStream_t st);
int resident_dispatch_electrode(const tf_resident& p, const ResidentArgs& a, int periodic, hipStream_t st);
int resident_dispatch_field(const tf_resident& p, const ResidentArgs& a, hipStream_t st);
int resident_dispatch_mpfaces(const tf_resident& p, const ResidentArgs& a, hipStream_t st);
