// The chunk walk on 32-token chunks with a 4-wave workgroup (included by prefill.hip, inside its namespace).
//
// chunk_kernel keeps a 64-token chunk's operands in 158 KiB of LDS, so a CU holds one workgroup: its 8 waves (two
// per SIMD) meet at the same four barriers per chunk and stall together.  Here a chunk is 32 tokens, the row arrays
// halve and the workgroup needs 75.2 KiB, so two independent workgroups share a CU: still two waves per SIMD, but from
// workgroups whose barriers and dependent chains do not line up.  Per token the work is the same (the Gram and solve
// blocks shrink with the chunk; the per-chunk state work -- decay, fp16 copies of S -- doubles).  Each wave keeps a
// 128 x 32 slice of S (64 VGPRs), so a piece that also carries its transition does not fit: this kernel runs unsplit
// layouts only: the plan picks it (KdaPrefillPlan.chunk32) for layouts whose items outnumber the CUs when its schedule
// model has it finish first, and launches in the precise mode keep chunk_kernel.
//
// Same algorithm, phases and operand conventions as chunk_kernel, with two row blocks of 16 instead of four:
//   P0-P2 rows to gated operands in registers (chunk_front), then the 7 block-factor rows, P4 Gram tiles (wave I = 0
//   / 1: diagonal block I's A_kk with the bf16 hi / lo split, then T_II; wave 2 + I: its A_qk, then one product of
//   block (1, 0)), P5 Q~ and Kd^T layouts (tokens permuted by pos32),
//   P6 W / U (wave w: channel / value tiles 2 w, 2 w + 1),
//   P7 the walk (wave w: S[:, 32 w .. 32 w + 31], K step outermost).  Checkpoints fall on 64-token boundaries, i.e.
//   after every second chunk (or after the last chunk of the sequence).
constexpr int C32_THREADS = 256;
constexpr int RST32 = 48;                                // rows of 32 tokens (fp16): 6 slots, no conflicts (see RST)
constexpr int RSV32 = 40;                                // V^T rows (bf16, 32 tokens)
constexpr int RSA32 = 40;                                // -A_kk / T_II rows
constexpr int W_HALF32 = 32 * RSW;                       // elements of a half array of W
constexpr int C32_A = 0;                                 // k^ fi: fp32 [32][RS32]
constexpr int C32_B = C32_A + 32 * RS32 * 4;             // q^ fi fp32 [32][RS32]; then Q~ fp16 [32][RSQ]
constexpr int C32_BV = C32_B + 32 * RSQ * 2;             // -W fp16 [2][32][RSW] (region B's upper half)
constexpr int C32_C = C32_BV + 2 * W_HALF32 * 2;         // k^ fj fp32 [32][RS32]; then Kd^T fp16 [128][RST32]
constexpr int C32_VT = C32_C + 32 * RS32 * 4;            // V^T bf16 [128][RSV32]
constexpr int C32_AQ = C32_VT + 128 * RSV32 * 2;         // A_qk fp16 [32][RST32] (columns permuted)
constexpr int C32_AK = C32_AQ + 32 * RST32 * 2;          // -A_kk block (1, 0) and T_II diagonal blocks fp16 [32][RSA32]
constexpr int C32_F = C32_AK + 32 * RSA32 * 2;           // factor rows [7][RSF] fp32
constexpr int C32_WT = C32_F + 7 * RSF * 4;              // gate totals of the 4 waves' rows [4][128] fp32
constexpr int C32_BETA = C32_WT + 4 * 128 * 4;           // [32] fp32
constexpr int C32_DT = C32_BETA + 32 * 4;                // An dt_bias [128] fp32 (gate in the kernel)
constexpr int C32_L = C32_DT + 128 * 4;                  // -L_II diagonal blocks, column-major [2][16][20] fp32
constexpr int C32_TOTAL = C32_L + 2 * 16 * 20 * 4;
static_assert(32 * RS32 * 4 <= 32 * RSQ * 2 + 2 * W_HALF32 * 2, "q^ fi fits region B");
static_assert(128 * RST32 * 2 <= 32 * RS32 * 4, "Kd^T fits region C");
static_assert(W_HALF32 * 2 % 256 == 0, "half arrays share their banks");
static_assert(2 * C32_TOTAL <= 160 * 1024, "two workgroups per CU");
// factor rows: a_1 = e^{Gamma_m(1) - Gamma_15}, b_10 = e^{Gamma_15 - Gamma_m(0)}, x_I = e^{Gamma_m(I)},
// y_I = e^{Gamma_c - Gamma_m(I)}, e^{Gamma_c} (Gamma_m(I): the middle row 16 I + 7 of block I; Gamma_c: the last row)
constexpr int F32_A = 0, F32_B = 1, F32_X = 2, F32_Y = 4, F32_DEC = 6;

// S slice of this lane (k = 16 dt + 4 g .. + 3, v = 32 w + 16 ct + m) to a V-major [128][128] fp32 / bf16 state
__device__ __forceinline__ void store_state32(float* dst, const f32x4 (&S)[8][2], int w, int g, int m) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        float* row = dst + (32 * w + 16 * ct + m) * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<f32x4*>(row + 16 * dt) = S[dt][ct];
    }
}
__device__ __forceinline__ void store_state32_bf16(uint16_t* dst, const f32x4 (&S)[8][2], int w, int g, int m) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        uint16_t* row = dst + (32 * w + 16 * ct + m) * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
            *reinterpret_cast<u32x2*>(row + 16 * dt) =
                u32x2{f2bf2(S[dt][ct][0], S[dt][ct][1]), f2bf2(S[dt][ct][2], S[dt][ct][3])};
    }
}

template <bool RG>
__global__ void __launch_bounds__(C32_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
    chunk32_kernel(PfParams p, const int32_t* __restrict__ tab, const int32_t* __restrict__ ck_idx, int list_off) {
    extern __shared__ __align__(16) unsigned char lds[];
    float* sKA = reinterpret_cast<float*>(lds + C32_A);
    float* sQA = reinterpret_cast<float*>(lds + C32_B);
    half_t* sQt = reinterpret_cast<half_t*>(lds + C32_B);
    half_t* sW = reinterpret_cast<half_t*>(lds + C32_BV);
    float* sKB = reinterpret_cast<float*>(lds + C32_C);
    half_t* sKd = reinterpret_cast<half_t*>(lds + C32_C);
    uint16_t* sVt = reinterpret_cast<uint16_t*>(lds + C32_VT);
    half_t* sAq = reinterpret_cast<half_t*>(lds + C32_AQ);
    half_t* sAk = reinterpret_cast<half_t*>(lds + C32_AK);
    float* sL = reinterpret_cast<float*>(lds + C32_L);
    float* sF = reinterpret_cast<float*>(lds + C32_F);
    float* sWt = reinterpret_cast<float*>(lds + C32_WT);
    float* sBeta = reinterpret_cast<float*>(lds + C32_BETA);
    float* sDT = reinterpret_cast<float*>(lds + C32_DT);

    const int H = p.H;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    const bool pool = (p.flags & KDA355_PF_POOL) != 0;
    const bool RB = (p.flags & KDA355_PF_RAW_BETA) != 0;
    const bool NORM = (p.flags & KDA355_PF_NORMALIZE_QK) != 0;
    const int ck_mode = (p.flags & KDA355_PF_CK_EVERY) ? 2 : ((p.flags & KDA355_PF_CK_SINGLE) ? 1 : 0);
    const int every = tab[H_EVERY];
    // one (chain entry, head) item per workgroup; an unsplit layout's entries are whole sequences
    const int item = (int)blockIdx.x;
    const int ci = item / H;
    const int h = item - ci * H;
    const int32_t* en = tab + list_off + C_WORDS * ci;
    const int n = en[C_SEQ], tstart = en[C_TSTART], len = en[C_LEN], pflags = en[C_FLAGS];
    const int first = en[C_FIRST], seqch = en[C_SEQCH], ck_row0 = en[C_CKROW0];
    const int ck_single = (ck_mode == 1) ? en[C_CKSINGLE] : 0;
    const int nch = (len + 31) >> 5;
    int64_t prow = -1;
    const float* src = nullptr;
    if (pool) {
        prow = p.state_idx[n];
        src = (prow >= 0 && prow < p.state_slots && p.has_init[n] != 0)
                  ? p.state_pool + prow * p.state_ss + (int64_t)h * D * D : nullptr;
    } else {
        src = p.init_state ? p.init_state + ((int64_t)n * H + h) * D * D : nullptr;
    }
    int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
    int c4 = lane & 31, row0 = 8 * w + 4 * (lane >> 5);  // the lane's channels 4 c4 .. + 3 and rows row0 .. + 3
    const float dtb = RG ? p.dt_bias[h * D + (tid & (D - 1))] : 0.f;
    const float alog = RG ? p.A_log[h] : 0.f;
    RawRows<RG> nx;
    load_rows<RG>(p, h, tstart, nch > 0 ? min(32, len) : 0, row0, c4, RB, nx);  // an empty sequence loads nothing
    f32x4 S[8][2];
    {
        // through a descriptor of no records when there is no start state; base and size wave-uniform
        const int nrec = __builtin_amdgcn_readfirstlane(src ? D * D * 4 : 0);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            uniform_ptr(src ? static_cast<const void*>(src) : static_cast<const void*>(p.q)), (short)0, nrec, 0x00020000);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const int voff = ((32 * w + 16 * ct + m) * D + 4 * g) * 4;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
                S[dt][ct] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff + 64 * dt, 0, 0));
        }
    }
    auto ck_store = [&](int64_t rr) {
        if (rr < 0 || rr >= p.ck_slots) return;
        if (p.ck_bf16)
            store_state32_bf16(reinterpret_cast<uint16_t*>(p.ck_pool) + rr * p.ck_ss + (int64_t)h * D * D, S, w, g, m);
        else
            store_state32(reinterpret_cast<float*>(p.ck_pool) + rr * p.ck_ss + (int64_t)h * D * D, S, w, g, m);
    };
    float An = 0.f;
    if (RG) {
        An = gate_an(alog);
        if (tid < D) sDT[tid] = An * dtb;
    }
    // A_qk block (0, 1) is read by the walk and never written by the Gram phase
    sAq[(tid >> 4) * RST32 + pos32(16 + (tid & 15))] = (half_t)0.f;
    lds_barrier();

    for (int cl = 0; cl < nch; ++cl) {
        // lane indices re-derived every chunk from an opaque copy (recomputed where used, not kept live)
        tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        lane = tid & 63;
        m = lane & 15;
        g = lane >> 4;
        c4 = lane & 31;
        row0 = 8 * w + 4 * (lane >> 5);
        const int t0 = tstart + 32 * cl, L = min(32, len - 32 * cl);
        const bool pf = cl + 1 < nch;
        const int pf_t = t0 + 32, pf_L = pf ? min(32, len - 32 * (cl + 1)) : 0;
        // ================= P0-P2: the wave's rows to gated operands in registers, then to regions A, B, C; block factors
        f32x4 kfj[4], qfi[4];
        {
            f32x4 kfi[4];
            chunk_front<RG>(nx, w, lane, L, RB, NORM, An, p.lb, sDT, sWt, sBeta, sVt, RSV32, kfi, kfj, qfi);
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4*>(&sKA[(row0 + j) * RS32 + 4 * c4]) = kfi[j];
            lds_barrier();
        }
        {
            const int c = tid & 127, qd = __builtin_amdgcn_readfirstlane(tid >> 7);  // wave-uniform
            const int fc = f_at(c);
            // gate totals of rows 8 i .. 8 i + 7; Gamma at rows 7, 15, 23, 31 are their running sums
            const float t0 = sWt[c], t1 = sWt[128 + c], t2 = sWt[256 + c], t3 = sWt[384 + c];
            if (qd == 0) {
                sF[F32_A * RSF + fc] = exp2_(t2);
                sF[F32_X * RSF + fc] = exp2_(t0);
                sF[(F32_Y + 1) * RSF + fc] = exp2_(t3);
                sF[F32_DEC * RSF + fc] = exp2_((t0 + t1) + (t2 + t3));
            } else {
                sF[F32_B * RSF + fc] = exp2_(t1);
                sF[(F32_X + 1) * RSF + fc] = exp2_((t0 + t1) + t2);
                sF[F32_Y * RSF + fc] = exp2_(t1 + (t2 + t3));
            }
        }
        // after the factors, whose reads of the gate totals would otherwise queue behind these writes in the LDS (with the
        // lane's q^ fi and k^ fj held to the layouts instead of read back: 32 x 512 tokens, H 12, 122 -> 119 us)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int o = (row0 + j) * RS32 + 4 * c4;
            *reinterpret_cast<f32x4*>(&sKB[o]) = kfj[j];
            *reinterpret_cast<f32x4*>(&sQA[o]) = qfi[j];
        }
        load_rows_qk(p, h, pf_t, pf_L, row0, c4, nx, 1);  // the next chunk's rows, one group a phase (see load_rows_qk)
        lds_barrier();
        load_rows_qk(p, h, pf_t, pf_L, row0, c4, nx, 2);
        // ================= P4: Gram tiles.  Wave I (0, 1): the diagonal block's A_kk (bf16 hi + lo products of
        // k^ fi and k^ fj), then T_II = (I + L_II)^-1; wave 2 + I: the same block's A_qk (k^ fj and q^ fi), then one
        // product of block (1, 0) from fp16 operands <= 1 (reference row 15): A_kk on wave 2, A_qk on wave 3.
        {
            const int I = w & 1, i = 16 * I + m;
            const bool kk = w < 2;  // wave-uniform
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            const float* sX = kk ? sKA : sQA;  // the product's second operand: k^ fi (A_kk) or q^ fi (A_qk)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c0 = gram_c0(s, g);
                uint32_t xh[4], xl[4], kbh[4], kbl[4];
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const f32x4 xa = *reinterpret_cast<const f32x4*>(&sX[i * RS32 + c0 + 4 * hf]);
                    const f32x4 kb = *reinterpret_cast<const f32x4*>(&sKB[i * RS32 + c0 + 4 * hf]);
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int ee = 2 * hf + j;
                        split_bf16x2(xa[2 * j], xa[2 * j + 1], xh[ee], xl[ee]);
                        split_bf16x2(kb[2 * j], kb[2 * j + 1], kbh[ee], kbl[ee]);
                    }
                }
                const bf16x8 Xh = as_bf16x8(xh), Xl = as_bf16x8(xl), Kbh = as_bf16x8(kbh), Kbl = as_bf16x8(kbl);
                if (kk) {  // A_kk: lane (g, m) holds row 16 I + 4 g + e, column 16 I + m
                    acc = mfma32bf(Xh, Kbh, acc);
                    acc = mfma32bf(Xh, Kbl, acc);
                    acc = mfma32bf(Xl, Kbh, acc);
                } else {   // A_qk transposed: lane (g, m) holds row 16 I + m, columns 16 I + 4 g .. + 3
                    acc = mfma32bf(Kbh, Xh, acc);
                    acc = mfma32bf(Kbl, Xh, acc);
                    acc = mfma32bf(Kbh, Xl, acc);
                }
            }
            if (kk) {
                f32x4 lt;
                const f32x4 bt4 = *reinterpret_cast<const f32x4*>(&sBeta[16 * I + 4 * g]);
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) lt[ee] = (m < 4 * g + ee) ? -(bt4[ee] * acc[ee]) : 0.f;
                *reinterpret_cast<f32x4*>(&sL[(I * 16 + m) * 20 + 4 * g]) = lt;
                const f32x4 x = invert_unit_lower(sL + I * 16 * 20, g, m);
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) sAk[(16 * I + 4 * g + ee) * RSA32 + 16 * I + m] = (half_t)x[ee];
            } else {
                f16x4 aq;
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) aq[ee] = (half_t)((4 * g + ee <= m) ? acc[ee] : 0.f);  // causal
                *reinterpret_cast<f16x4*>(&sAq[i * RST32 + pos32(16 * I + 4 * g)]) = aq;
            }
        }
        if (w >= 2) {  // block (1, 0): wave 2 A_kk, wave 3 A_qk (transposed tiles: lane (g, m) holds row 16 + m,
                       // columns 4 g .. + 3)
            const bool kk = w == 2;
            const int i = 16 + m;
            const float* sX = kk ? sKA : sQA;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c0 = gram_c0(s, g);
                f16x8 xa, kb;
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const f32x4 a = *reinterpret_cast<const f32x4*>(&sX[i * RS32 + c0 + 4 * hf]);
                    const f32x4 fa = *reinterpret_cast<const f32x4*>(&sF[F32_A * RSF + f_at(c0) + 4 * hf]);
                    const f32x4 b = *reinterpret_cast<const f32x4*>(&sKB[m * RS32 + c0 + 4 * hf]);
                    const f32x4 fb = *reinterpret_cast<const f32x4*>(&sF[F32_B * RSF + f_at(c0) + 4 * hf]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        xa[4 * hf + j] = (half_t)(a[j] * fa[j]);
                        kb[4 * hf + j] = (half_t)(b[j] * fb[j]);
                    }
                }
                acc = mfma32(kb, xa, acc);
            }
            if (kk) {
                const float nb = -sBeta[i];
                f16x4 ak;
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) ak[ee] = (half_t)(nb * acc[ee]);
                *reinterpret_cast<f16x4*>(&sAk[i * RSA32 + 4 * g]) = ak;
            } else {
                f16x4 aq;
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) aq[ee] = (half_t)acc[ee];
                *reinterpret_cast<f16x4*>(&sAq[i * RST32 + pos32(4 * g)]) = aq;
            }
        }
        // ================= P5: Q~, Kd^T into their walk layouts (the lane's rows)
        // the start state's loads complete here in the first chunk (an empty use of S), not before a later walk
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) asm volatile("" : "+v"(S[dt][ct]));
        load_rows_vb(p, h, pf_t, pf_L, row0, c4, RB, nx);
        lds_barrier();  // regions B and C are rewritten below
        {
            const f32x4 xf = *reinterpret_cast<const f32x4*>(&sF[(F32_X + (w >> 1)) * RSF + f_at(4 * c4)]);
            const f32x4 yf = *reinterpret_cast<const f32x4*>(&sF[(F32_Y + (w >> 1)) * RSF + f_at(4 * c4)]);
            const int qc = 32 * (c4 >> 3) + 8 * (c4 & 3) + (c4 & 4);  // stored position of channel 4 c4
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f16x4 o;
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) o[ee] = (half_t)(qfi[j][ee] * xf[ee]);
                *reinterpret_cast<f16x4*>(&sQt[(row0 + j) * RSQ + qc]) = o;
            }
            const int pr = pos32(row0);  // stored position of token row0 (row0 + 1 .. 3 follow it)
#pragma unroll
            for (int ee = 0; ee < 4; ++ee) {
                f16x4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = (half_t)(kfj[j][ee] * yf[ee]);
                *reinterpret_cast<f16x4*>(&sKd[ch_row(4 * c4 + ee) * RST32 + pr]) = o;
            }
        }
        // ================= P6: W and U by block forward substitution (wave w: channel / value tiles 2 w, 2 w + 1)
        load_rows_g<RG>(p, h, pf_t, pf_L, row0, c4, nx);
        f32x4 Ur[2][2];  // [block I][tile t]: U[token 16 I + 4 g + e][value 32 w + 16 t + m]
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int tw = 2 * w + t, c = 16 * tw + m;
            f16x4 Xh0, Uh0;
#pragma unroll
            for (int I = 0; I < 2; ++I) {
                const float xI = sF[(F32_X + I) * RSF + f_at(16 * tw) + m];
                const f32x4 b4 = *reinterpret_cast<const f32x4*>(&sBeta[16 * I + 4 * g]);
                const u32x2 v4 = *reinterpret_cast<const u32x2*>(&sVt[(16 * tw + (m ^ tw)) * RSV32 + 16 * I + 4 * g]);
                const float vf[4] = {bf2f(v4.x & 0xffffu), bf2f(v4.x >> 16), bf2f(v4.y & 0xffffu), bf2f(v4.y >> 16)};
                f32x4 aw, au;
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) {
                    aw[ee] = b4[ee] * sKA[(16 * I + 4 * g + ee) * RS32 + c] * xI;
                    au[ee] = b4[ee] * vf[ee];
                }
                if (I == 1) {
                    const f16x4 A = *reinterpret_cast<const f16x4*>(&sAk[(16 + m) * RSA32 + 4 * g]);
                    aw = mfma16(A, Xh0, aw);
                    au = mfma16(A, Uh0, au);
                }
                const f16x4 T = *reinterpret_cast<const f16x4*>(&sAk[(16 * I + m) * RSA32 + 16 * I + 4 * g]);
                f16x4 bwh, buh;
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) { bwh[ee] = (half_t)aw[ee]; buh[ee] = (half_t)au[ee]; }
                const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                // W's tile transposed (see chunk_kernel): 4 consecutive channels of token 16 I + m per lane
                const f32x4 Xt = mfma16(bwh, T, z);
                Ur[I][t] = mfma16(T, buh, z);
                *reinterpret_cast<f16x4*>(&sW[half_at(16 * I + m, 32 * w + 8 * g + 4 * t, RSW, W_HALF32)]) =
                    f16x4{(half_t)-Xt[0], (half_t)-Xt[1], (half_t)-Xt[2], (half_t)-Xt[3]};
                if (I == 0) {
                    const f32x4 Xw = mfma16(T, bwh, z);
#pragma unroll
                    for (int ee = 0; ee < 4; ++ee) { Xh0[ee] = (half_t)Xw[ee]; Uh0[ee] = (half_t)Ur[0][t][ee]; }
                }
            }
        }
        lds_barrier();
        // ================= P7: the walk (wave w: S[:, 32 w .. 32 w + 31])
        // every-n row 0: the state before the sequence's first token
        if (cl == 0 && ck_mode == 2 && every > 0 && first == 0) ck_store(ck_idx[ck_row0]);
        {
            f16x8 SB[4][2];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for (int ee = 0; ee < 4; ++ee) {
                        SB[s][ct][ee] = (half_t)S[2 * s][ct][ee];
                        SB[s][ct][4 + ee] = (half_t)S[2 * s + 1][ct][ee];
                    }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int it = 0; it < 2; ++it) {
                    const f16x8 A = *reinterpret_cast<const f16x8*>(&sW[half_at(16 * it + m, 32 * s + 8 * g, RSW, W_HALF32)]);
#pragma unroll
                    for (int ct = 0; ct < 2; ++ct) Ur[it][ct] = mfma32(A, SB[s][ct], Ur[it][ct]);
                }
            f16x8 VB[2];  // V' = U - W S (accumulated onto U: sW holds -W) as fp16, tokens 4 g + e and 16 + 4 g + e
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int ee = 0; ee < 4; ++ee) {
                    VB[ct][ee] = (half_t)Ur[0][ct][ee];
                    VB[ct][4 + ee] = (half_t)Ur[1][ct][ee];
                }
            // O^T = S^T Q~^T + V'^T A_qk^T (lane (g, m): token 16 it + m, values 32 w + 16 ct + 4 g .. + 3)
            f32x4 ao[2][2];
#pragma unroll
            for (int it = 0; it < 2; ++it)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) ao[it][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int it = 0; it < 2; ++it) {
                    const f16x8 B = *reinterpret_cast<const f16x8*>(&sQt[(16 * it + m) * RSQ + 32 * s + 8 * g]);
#pragma unroll
                    for (int ct = 0; ct < 2; ++ct) ao[it][ct] = mfma32(SB[s][ct], B, ao[it][ct]);
                }
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const f16x8 B = *reinterpret_cast<const f16x8*>(&sAq[(16 * it + m) * RST32 + 8 * g]);
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) ao[it][ct] = mfma32(VB[ct], B, ao[it][ct]);
            }
#pragma unroll
            for (int it = 0; it < 2; ++it)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) {
                    const u32x2 o = {f2bf2(p.scale * ao[it][ct][0], p.scale * ao[it][ct][1]),
                                     f2bf2(p.scale * ao[it][ct][2], p.scale * ao[it][ct][3])};
                    if (16 * it + m < L)
                        *reinterpret_cast<u32x2*>(p.out + ((int64_t)t0 + 16 * it + m) * p.out_rs + (int64_t)h * D +
                                                  32 * w + 16 * ct + 4 * g) = o;
                }
            // S <- diag(e^{Gamma_c}) S + Kd^T V'
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                const f32x4 d4 = *reinterpret_cast<const f32x4*>(&sF[F32_DEC * RSF + f_at(16 * dt) + 4 * g]);
                const f16x8 A = *reinterpret_cast<const f16x8*>(&sKd[(16 * dt + (m ^ dt)) * RST32 + 8 * g]);
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) {
#pragma unroll
                    for (int ee = 0; ee < 4; ++ee) S[dt][ct][ee] *= d4[ee];
                    S[dt][ct] = mfma32(A, VB[ct], S[dt][ct]);
                }
            }
        }
        // checkpoints at 64-token boundaries: after every second chunk, and after the sequence's last chunk
        if ((cl & 1) || cl + 1 == nch) {
            const int cs = first + ((cl + 2) >> 1);
            if (ck_mode == 1 && cs == ck_single) ck_store(ck_idx[n]);
            if (ck_mode == 2 && every > 0 && cs % every == 0 && cs < seqch) ck_store(ck_idx[ck_row0 + cs / every]);
        }
        // no barrier here: the walk writes no LDS and reads nothing the next chunk writes before its first barrier
    }
    if (pflags & PIECE_LAST) {
        if (pool) {
            if (prow >= 0 && prow < p.state_slots) store_state32(p.state_pool + prow * p.state_ss + (int64_t)h * D * D, S, w, g, m);
        } else {
            store_state32(p.final_state + ((int64_t)n * H + h) * D * D, S, w, g, m);
        }
    }
}

template <bool RG>
hipError_t launch_chunk32(const PfParams& p, int list_off, int wgs, hipStream_t s) {
    static bool attr_set = false;  // idempotent; a race only repeats the call
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(chunk32_kernel<RG>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, C32_TOTAL);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL((chunk32_kernel<RG>), dim3(wgs), dim3(C32_THREADS), C32_TOTAL, s, p, p.tab, p.ck_idx, list_off);
    return hipGetLastError();
}
