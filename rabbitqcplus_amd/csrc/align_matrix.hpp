// Shifted-Hamming alignment with the matrix cores as a filter (included by care_hip.hip
// inside its anonymous namespace).
//
// The alignment wants, per candidate and orientation, the admissible shift of minimum
// (score, scan index) (the argmin that alignBoth states). Nearly every shift of a read pair
// is hopeless: an admissible one has fewer than int(overlap * maxErrorRate) mismatches,
// random sequence has 3/4 of the overlap. So the scan is split in two:
//
//  filter   the mismatches of the lo plane alone (purine / pyrimidine: A,G against C,T) are
//           a lower bound of the mismatches. With lo bits as +1 / -1 and 0 outside a read,
//           overlap - 2 * loMismatches of every shift is a Toeplitz matrix product: rows =
//           32 consecutive shifts of the anchor, columns = 16 candidates x 2 orientations,
//           depth = 64 candidate positions per v_mfma_f32_32x32x64_f8f6f4 with fp4 operands
//           (+-1 and 0 are exact in fp4, sums of at most 1024 of them exact in fp32). The
//           accumulator starts at minus the least value an admissible shift can have, so a
//           shift passes iff its sign bit is 0. Zeros outside the reads do the overlap masks.
//  exact    the few shifts that pass (about one per candidate, its true one) go through a
//           queue in LDS and are counted exactly on both planes, two lanes per shift; the
//           (score, scan index) minimum per candidate and orientation is an LDS minimum.
//
// Results are those of the scan for every input: the filter passes every admissible shift,
// whatever order they are counted in. Reads of low complexity pass many shifts; an anchor
// whose queue takes more than kMatrixBudget per candidate so far (of 16 at least, which ends
// most of them in their first block, before anything is counted) is listed and redone by a scan
// (lane per candidate, or for reads of more than 352 bases wavefront per pair), which costs
// about the same for any sequence: an exact count costs some 4 instructions per shift, the
// scan of every shift some 150 per candidate. Alignment of reads that are 90% tandem repeats
// of one or two bases, against the scan alone: 1.13 against 1.28 ms (80,000 of 150 bases), 2.1
// against 2.35 (68,571 of 100..250), 7.8 against 7.7 (18,461 of 600..700).
//
// Measured (MI355X): 1.0M x 150 bases 12.15 -> 4.6 ms against the lane scan, 1.03M reads of
// 100..250 bases 28.8 -> 8.5 ms, 60,000 of 360..450 bases 7.4 -> 1.2 ms against the wavefront
// per pair. At 150 bases: 3.1k vector and 1.6k scalar instructions per anchor (1.1 and 0.6
// per clock and CU at 5.8 waves per SIMD), matrix cores busy a fifth of the time; bound by
// instruction issue and by the latency of its LDS and accumulator reads.
//
// Position order inside a 64-deep step is free as long as both operands share it: dword i
// of a lane's 32 positions holds positions 4n + i in nibbles n, so a nibble dword is one
// shift and one and-or from a plane word, and the anchor's dword i at bit offset o is its
// dword 0 at offset o + i: one LDS dword per bit offset feeds the whole Toeplitz matrix
// (a lane reads four consecutive ones; 4.7 KB of LDS per wave at 150 bases, where 16-byte
// fragments took 7.9 KB and held the kernel at 4.3 waves per SIMD).

typedef int MatrixFrag __attribute__((ext_vector_type(8)));
typedef float MatrixAcc __attribute__((ext_vector_type(16)));
typedef uint32_t Words4 __attribute__((ext_vector_type(4)));

constexpr int kMatrixCands = 16;        // candidates per column block (x 2 orientations)
constexpr int kMatrixQueue = 192;       // queued shifts; counted when fewer than 64 free
constexpr int kMatrixBudget = 8;        // queued shifts per candidate before an anchor is listed
constexpr float kMatrixMaxRate = 0.3f;  // error rates up to which the lo plane separates shifts well
constexpr int kMatrixMinShifts = 12;    // shifts per direction from which the filter pays

// LDS layout in dwords for planes of W words: anchor word pairs (hi, lo), anchor nibbles,
// candidate rows of one block, queue, per-candidate keys and lengths of a 64-candidate chunk.
struct MatrixLds {
    int frag, rows, rowStride, queue, keys, lens, bytes;
};
__host__ __device__ inline MatrixLds matrixLds(int W){
    MatrixLds l;
    const int pairs = 2 * 2 * (W + 6);              // uint2 per word index -4..W+1, two planes
    l.frag = (pairs + 3) & ~3;
    l.rows = l.frag + (W + 6) * 32 + 4;             // bit offsets from word -4 on
    l.rowStride = 4 * W + 4;                        // 16 bytes of padding against bank conflicts
    l.queue = l.rows + kMatrixCands * l.rowStride;
    l.keys = l.queue + kMatrixQueue;
    l.lens = l.keys + 2 * kWave;
    l.bytes = (l.lens + kWave) * 4;
    return l;
}

// +-1 / 0 as fp4 nibbles of dword i: value bits v, validity bits m (v is 0 where m is 0)
__device__ __forceinline__ int signNibbles(uint32_t v, uint32_t m, int i){
    const uint32_t one = i < 2 ? m >> (2 - i) : m << (i - 2);
    return int(((v << i) & 0x88888888u) | (one & 0x22222222u));
}

// Larger of x and a negative y as floats: with y's sign bit set, the smaller bit pattern (no
// NaN quieting, which costs fmaxf a second instruction per operand)
__device__ __forceinline__ float maxNegative(float x, float y){
    return __uint_as_float(min(__float_as_uint(x), __float_as_uint(y)));
}

// Least and largest value over the 16 lanes of a row (DPP: neighbours, pairs, mirrored halves).
__device__ __forceinline__ void rowMinMax(int& lo, int& hi){
#define ROW_STEP(ctrl) \
    lo = min(lo, __builtin_amdgcn_update_dpp(lo, lo, ctrl, 0xf, 0xf, false)); \
    hi = max(hi, __builtin_amdgcn_update_dpp(hi, hi, ctrl, 0xf, 0xf, false));
    ROW_STEP(0xB1) ROW_STEP(0x4E) ROW_STEP(0x141) ROW_STEP(0x140)     // quad_perm 1,0,3,2 / 2,3,0,1, half mirror, mirror
#undef ROW_STEP
}

template<int KB>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(KB <= 3 ? 6 : (KB <= 4 ? 5 : (KB <= 6 ? 4 : 2)))))
k_align_matrix(AlignParams p){
    extern __shared__ __align__(16) uint32_t lds[];
    if(int(blockIdx.x) >= p.B) return;
    const int ai = batchAnchor(p.order, p.B);
    const uint32_t beg = p.offsets[ai];
    const int n = int(p.offsets[ai + 1] - beg);
    if(n == 0) return;
    const int lane = threadIdx.x;
    const int W = p.W;
    const MatrixLds L = matrixLds(W);
    uint2* const aPair = reinterpret_cast<uint2*>(lds);         // [plane][word + 4] = (word + 1, word)
    const int pairs = W + 6;
    uint32_t* const frag = lds + L.frag;
    uint32_t* const rows = lds + L.rows;
    uint32_t* const queue = lds + L.queue;
    uint32_t* const keys = lds + L.keys;
    int* const lens = reinterpret_cast<int*>(lds + L.lens);

    const uint64_t a = p.b0 + uint64_t(ai);
    const int La = p.len[a];
    const uint32_t* arow = p.hilo + a * uint64_t(4 * W);
    // first candidates' ids, on the way while the anchor is prepared
    uint32_t id = lane < n ? p.ids[beg + uint32_t(lane)] : 0u;
    int Lc = lane < n ? p.len[id] : 0;

    for(int q = lane; q < 2 * pairs; q += kWave){
        const int pl = q >= pairs ? 1 : 0;
        const int w = q - pl * pairs - 4;
        const uint32_t w0 = (w >= 0 && w < W) ? arow[pl * W + w] : 0u;
        const uint32_t w1 = (w + 1 >= 0 && w + 1 < W) ? arow[pl * W + w + 1] : 0u;
        aPair[q] = make_uint2(w1, w0);
    }
    __syncthreads();

    // scanned shifts: 0..La-mo and -1..-(Lc-mo). Blocks of 32 shifts end at the last one.
    const int mo = max(max(p.minOverlap, int(float(La) * p.minOverlapRatio)), 1);
    const int F = max(La - mo + 1, 0);                  // scan index of shift -1
    const int sTop = F - 1;                             // -1 when the anchor is too short to be shifted
    const int sAlign = sTop + 1;                        // blocks start at sAlign - 32 * k
    const int delta = sAlign & 31;
    const int Wa = (La + 31) >> 5;
    // nibble dword 0 of the 32 anchor positions from bit offset 32 * -4 + delta + q (all zero in
    // words -4, -3 of the first half's and W, W + 1 of the second half's rows)
    for(int q = lane; q < (W + 6) * 32 + 4; q += kWave){
        const int o = q - 128 + delta;
        const uint2 pr = aPair[pairs + min(max(((o + 31) >> 5) + 3, 0), pairs - 1)];
        const uint32_t v = __builtin_amdgcn_alignbit(pr.y, pr.x, uint32_t(-o) & 31u);
        const uint32_t m = overlapMask(La - o) & ~overlapMask(-o);
        frag[q] = uint32_t(signNibbles(v & m, m, 0));
    }

    const int half = lane >> 5;
    const int col = lane & 31;
    const int orient = (lane >> 4) & 1;
    const float c1 = 1.0f - 2.0f * p.maxErrorRate;
    int counted = 0;                    // queued shifts so far
    auto giveUp = [&](){
        if(lane == 0){
            const ListedAnchors l(p, ai);
            l.ids[atomicAdd(l.count, 1u)] = uint32_t(ai);
        }
    };

    for(int c0 = 0; c0 < n; c0 += kWave){
        if(c0 > 0){
            id = c0 + lane < n ? p.ids[beg + uint32_t(c0 + lane)] : 0u;
            Lc = c0 + lane < n ? p.len[id] : 0;
        }
        const int cn = min(n - c0, kWave);
        __syncthreads();
        keys[lane] = 0xFFFFFFFFu;
        keys[kWave + lane] = 0xFFFFFFFFu;
        lens[lane] = Lc;
        const int nblocks = (cn + kMatrixCands - 1) / kMatrixCands;
        // rows of the next block, four lanes per candidate
        constexpr int NR = (2 * KB + 3) / 4;
        Words4 pre[NR] = {};
        auto fetch = [&](int b){
            const int c = b * kMatrixCands + (lane >> 2);
            const uint32_t rid = uint32_t(__shfl(int(id), c & 63));
            const Words4* src = reinterpret_cast<const Words4*>(p.hilo + uint64_t(rid) * uint64_t(4 * W));
            #pragma unroll
            for(int q = 0; q < NR; q++){
                const int ch = (lane & 3) + 4 * q;
                if(c < cn && ch < W) pre[q] = src[ch];
            }
        };
        fetch(0);
        for(int b = 0; b < nblocks; b++){
            __syncthreads();                            // the last block's rows are read no more
            {
                const int ci = lane >> 2;
                if(b * kMatrixCands + ci < cn){
                    Words4* dst = reinterpret_cast<Words4*>(rows + ci * L.rowStride);
                    #pragma unroll
                    for(int q = 0; q < NR; q++){
                        const int ch = (lane & 3) + 4 * q;
                        if(ch < W) dst[ch] = pre[q];
                    }
                }
            }
            if(b + 1 < nblocks) fetch(b + 1);
            __syncthreads();
            const int ci = b * kMatrixCands + (lane & 15);
            const bool cvalid = ci < cn;
            const int lc = cvalid ? lens[ci] : 0;
            // longest and shortest candidate of the block (wave-uniform)
            int lcMax = lc, lcMin = cvalid ? lc : INT_MAX;
            rowMinMax(lcMin, lcMax);
            lcMax = __builtin_amdgcn_readfirstlane(lcMax);
            lcMin = __builtin_amdgcn_readfirstlane(lcMin);
            // candidate fragments of this lane's column (no masks where every candidate of the block
            // covers the step's positions)
            MatrixFrag B[KB];
            {
                const uint32_t* lo = rows + (lane & 15) * L.rowStride + (orient ? 3 * W : W);
                #pragma unroll
                for(int kb = 0; kb < KB; kb++){
                    const int w = 2 * kb + half;
                    if(lcMin >= 64 * (kb + 1)){
                        const uint32_t v = lo[w];
                        B[kb] = MatrixFrag{signNibbles(v, ~0u, 0), signNibbles(v, ~0u, 1), signNibbles(v, ~0u, 2),
                                           signNibbles(v, ~0u, 3), 0, 0, 0, 0};
                    }else{
                        const uint32_t m = cvalid ? overlapMask(lc - 32 * w) : 0u;
                        const uint32_t v = m && w < W ? lo[w] & m : 0u;
                        B[kb] = MatrixFrag{signNibbles(v, m, 0), signNibbles(v, m, 1), signNibbles(v, m, 2),
                                           signNibbles(v, m, 3), 0, 0, 0, 0};
                    }
                }
            }
            const int nkb = (lcMax + 63) >> 6;
            const int lastB = max(lc - mo, 0);          // -lastB: most negative shift of this lane's candidate
            const int lastBMin = max(lcMin - mo, 0);
            const int sigma0 = -((sAlign + max(lcMax - mo, 0) + 31) >> 5);     // blocks sigma0..-1
            const float fLa = c1 * float(La), fLc = c1 * float(lc), fm = -c1 * float(min(La, lc)) - 1.5f;
            int qn = 0;
            // queued shifts that the candidates up to this block's last may have
            const int budget = max(min(c0 + (b + 1) * kMatrixCands, n), kMatrixCands) * kMatrixBudget;

            // counts the queued shifts exactly, two lanes per shift
            auto flush = [&](){
                __syncthreads();
                for(int e0 = 0; e0 < qn; e0 += 32){
                    const int e = e0 + (lane >> 1);
                    int mis = 0, s = 0, el = 0, eo = 0, ec = 0;
                    if(e < qn){
                        const uint32_t entry = queue[e];
                        s = int(entry >> 8) - 4096;
                        ec = int(entry & 15u);
                        eo = int(entry >> 4) & 1;
                        el = lens[b * kMatrixCands + ec];
                        const uint32_t* crow = rows + ec * L.rowStride + eo * 2 * W;
                        const int cbeg = max(-s, 0), cend = min(el, La - s);
                        for(int j = lane & 1; 32 * j < cend; j += 2){
                            const int lo = cbeg - 32 * j, hi = cend - 32 * j;   // hi > 0
                            if(lo < 32){
                                const uint32_t mask = (0xFFFFFFFFu >> max(lo, 0)) & (hi >= 32 ? ~0u : ~(0xFFFFFFFFu >> (hi & 31)));
                                const int o = 32 * j + s;               // in (-32, La)
                                const int at = ((o + 31) >> 5) + 3;     // words above and below the window's end
                                const uint2 vh = aPair[at], vl = aPair[pairs + at];
                                const uint32_t ah = __builtin_amdgcn_alignbit(vh.y, vh.x, uint32_t(-o) & 31u);
                                const uint32_t al = __builtin_amdgcn_alignbit(vl.y, vl.x, uint32_t(-o) & 31u);
                                mis += __popc(((ah ^ crow[j]) | (al ^ crow[W + j])) & mask);
                            }
                        }
                    }
                    mis += __builtin_amdgcn_update_dpp(0, mis, 0xB1, 0xf, 0xf, false);     // quad_perm 1,0,3,2
                    if(e < qn && (lane & 1) == 0){
                        const int ov = min(min(La - s, el + s), min(La, el));
                        if(mis < int(float(ov) * p.maxErrorRate)){
                            const int t = s >= 0 ? s : F - s - 1;
                            atomicMin(&keys[eo * kWave + b * kMatrixCands + ec],
                                      (uint32_t(mis + La + el - 2 * ov) << 16) | uint32_t(t));
                        }
                    }
                }
                qn = 0;
                __syncthreads();
            };

            // two blocks of 32 shifts per step: bits 0..15 and 16..31 of a lane's pass mask
            for(int sigma = sigma0; sigma < 0; sigma += 2){
                uint32_t pass = 0;
                #pragma unroll
                for(int u = 0; u < 2; u++){
                    if(sigma + u >= 0) break;
                    const int s0 = sAlign + 32 * (sigma + u);
                    const int xb = s0 >> 5;             // floor; delta is the rest
                    // the accumulators start at minus the least value an admissible shift
                    // can have, -(c1 * overlap + 1.5), overlap = min(La - s, lc + s, La, lc):
                    // one term for most blocks (wave-uniform tests)
                    MatrixAcc acc;
                    const float t0 = c1 * float(s0 + 4 * half);
                    const bool up = s0 >= 0;
                    const float base = up ? t0 - fLa - 1.5f : -t0 - fLc - 1.5f;
                    const float step = up ? c1 : -c1;
                    #pragma unroll
                    for(int i = 0; i < 16; i++) acc[i] = __builtin_fmaf(step, float((i & 3) + 8 * (i >> 2)), base);
                    if(up ? lcMin < La - s0 : (s0 + 31 > 0 || lcMax + s0 + 31 > La)){
                        #pragma unroll
                        for(int i = 0; i < 16; i++) acc[i] = maxNegative(acc[i], fm);
                        if(!up && s0 + 31 > 0){
                            #pragma unroll
                            for(int i = 0; i < 16; i++)
                                acc[i] = maxNegative(acc[i], __builtin_fmaf(c1, float((i & 3) + 8 * (i >> 2)), t0 - fLa - 1.5f));
                        }
                    }
                    #pragma unroll
                    for(int kb = 0; kb < KB; kb++){
                        const int x = xb + 2 * kb;      // word offset of this depth step's first half
                        // up to 3 steps run whether the anchor reaches them or not (x held in
                        // its zero words): a test and a branch per step cost more than the
                        // product, the scalar unit being nearly as busy as the vector unit
                        // (150 bases: 4.8 -> 4.6 ms; 4 steps on 100..250 bases: 8.5 -> 8.6 ms)
                        if(KB <= 3 || (kb < nkb && x >= -3 && x < Wa)){
                            const uint32_t* f = frag + (min(max(x, -4), W) + half + 4) * 32 + col;
                            const MatrixFrag A = {int(f[0]), int(f[1]), int(f[2]), int(f[3]), 0, 0, 0, 0};
                            acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B[kb], acc, 4, 4, 0, 0, 0, 0);
                        }
                    }
                    // sign bits: bit i of `miss` = row i of this lane does not pass
                    uint32_t miss = 0;
                    #pragma unroll
                    for(int i = 15; i >= 0; i--) miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(acc[i]), 31);
                    uint32_t in = 0xFFFFu;
                    if(s0 < -lastBMin){
                        // rows with shift >= -(Lc - mo); bit i <-> row (i & 3) + 8 * (i >> 2) + 4 * half
                        const int rmin = min(max(-lastB - s0, 0), 32);
                        in = uint32_t(0xFFFFFFFFull << rmin);
                        in = (in >> (4 * half)) & 0x0F0F0F0Fu;
                        in = (in | (in >> 4)) & 0x00FF00FFu;
                        in = (in | (in >> 8)) & 0xFFFFu;
                    }
                    pass |= (~miss & in) << (16 * u);
                }
                if(!cvalid) pass = 0;
                const int s0 = sAlign + 32 * sigma + 4 * half;
                for(;;){
                    const uint64_t any = __builtin_amdgcn_ballot_w64(pass != 0);
                    if(any == 0) break;
                    if(pass){
                        const int i = __builtin_ctz(pass);
                        pass &= pass - 1;
                        const int s = s0 + (i & 3) + 8 * (i >> 2);      // (bits 16.. are rows 32..)
                        const int at = qn + int(__builtin_amdgcn_mbcnt_hi(uint32_t(any >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(any), 0)));
                        queue[at] = (uint32_t(s + 4096) << 8) | uint32_t(col);
                    }
                    qn += int(__popcll(any));
                    if(qn > kMatrixQueue - kWave){
                        counted += qn;
                        if(counted > budget){ giveUp(); return; }
                        flush();
                    }
                }
            }
            counted += qn;
            if(counted > budget){ giveUp(); return; }
            if(qn) flush();
        }
        __syncthreads();
        if(lane < cn){
            const uint32_t kf = keys[lane], kr = keys[kWave + lane];
            OrientState sf, sr;
            sf.best = sr.best = La + Lc;
            if(kf != 0xFFFFFFFFu){ sf.best = int(kf >> 16); sf.bestT = int(kf & 0xFFFFu); }
            if(kr != 0xFFFFFFFFu){ sr.best = int(kr >> 16); sr.bestT = int(kr & 0xFFFFu); }
            const ShdResult f = finishOrientation(sf, La, Lc, F);
            const ShdResult rr = finishOrientation(sr, La, Lc, F);
            const int flag = chooseOrientation(f, rr, La, p);
            const ShdResult& sres = flag == 2 ? rr : f;
            AlignBest best;
            best.shift = sres.shift; best.overlap = sres.overlap; best.nOps = sres.nOps; best.orientation = flag;
            p.best[uint64_t(beg) + uint64_t(c0 + lane)] = best;
            if(p.dbg){
                int* d = p.dbg + (uint64_t(beg) + uint64_t(c0 + lane)) * 11;
                d[0] = f.score; d[1] = f.overlap; d[2] = f.shift; d[3] = f.nOps; d[4] = f.valid;
                d[5] = rr.score; d[6] = rr.overlap; d[7] = rr.shift; d[8] = rr.nOps; d[9] = rr.valid;
                d[10] = flag;
            }
        }
    }
}
