// Axis-by-axis form of the phase contraction on a regular mesh (included by
// elph_vertex.hip inside its anonymous namespace).
//
// The mesh drivers need Y(q) = sum_R e^{i 2 pi q.R} h(R) for (nearly) every q of
// an N0 x N1 x N2 mesh.  The exponential factors over the axes, so three short
// sums over one component of R each give the same Y as the product over all
// cells:
//   A  F1(q2; R0, R1) = sum_R2 e^{i 2 pi q2 R2 / N2} h(R)
//   B  F2(q2, q1; R0) = sum_R1 e^{i 2 pi q1 R1 / N1} F1(q2; R0, R1)
//   C  Y(q)           = sum_R0 e^{i 2 pi q0 R0 / N0} F2(q2, q1; R0)
// (axis_time weighs them against the product).  Axis 0 is the fastest index of the mesh,
// so the rows of one line (q1, q2) are consecutive rows of the driver's list and
// their results one contiguous range of the output.  Three kernels:
//   k_axis_rot   the band or branch rotation: h of the cells, in the order of the sums
//   k_axis_ab    A and B of 16 columns of one plane q2, F1 in LDS, F2 to memory
//   k_axis_pair / k_axis_pair_q   C and the epilogue of the driver, a wave per line
// B and C use the symmetric form: with C(q) = sum_R cos F+(R), S(q) = sum_R sin F-(R),
// F+- the sum and i times the difference of the terms of R and -R, the value at q is C + S
// and at -q C - S: real coefficients and half the q.
// Measured with 617 cells on 24^3, 8 bands, 6 branches (1786 states, 13824 rows): pair stage
// 53.0 ms per pass as one FP64 product (k_pair_fp64), 15.1 ms in int8 digits (k_pair_i8),
// 7.9 ms in this form (C and epilogue 5.2, A and B 2.1, rotation 0.6); ibzq (2478 states) 106 ms
// (k_pair_q_fp64) against 15.4 ms.  FP64 vector and matrix instructions share one pipe on this
// chip (their times add), so what is left is the epilogue's multiply-adds and its latency.

// Scalar (wave-uniform) loads.
typedef const __attribute__((address_space(4))) dv2 *sc_dv2;
typedef const __attribute__((address_space(4))) int *sc_int;
__device__ __forceinline__ sc_dv2 as_scalar(const double2 *p) { return (sc_dv2)(uintptr_t)p; }
__device__ __forceinline__ sc_int as_scalar(const int *p) { return (sc_int)(uintptr_t)p; }

template <int I>
using axis_int = std::integral_constant<int, I>;

// One cell list on one mesh, its cells by pairs (R0, R1) and R2 ("entries"), and the
// driver's rows by lines and planes.
struct AxisTab {
    int N0 = 1, N1 = 1, N2 = 1;
    int np = 0;                // pairs (R0, R1)
    int ncell = 0;             // entries (a multiple of 4 per pair: entries past a pair's cells are zero)
    int rm = 0, r1m = 0;       // largest |R0|, |R1|
    const int *pe = nullptr;           // [np + 1] first entry of a pair, most cells first
    const int *ecell = nullptr;        // [ncell] cell of an entry, -1 past a pair's cells
    const unsigned short *pidx = nullptr;  // [2 rm + 1][2 r1m + 1] pair of (R0, R1), np if there is none
    const double2 *phA = nullptr;      // [N2][ncell] e^{i 2 pi q2 R2 / N2}
    const double2 *T0 = nullptr, *T1 = nullptr;  // e^{i 2 pi j / N0}, e^{i 2 pi j / N1}
    // planes (one k2) and lines (one k1, k2) that hold rows; a launch takes npl planes from pl0 on and
    // their nl lines from l0 on, whose F2 it indexes from 0
    int npl = 0, nl = 0, pl0 = 0, l0 = 0;
    const int *pl_k2 = nullptr;        // [npl]
    const int *line_of = nullptr;      // [npl][N1] line of k1, -1 if it holds no row
    const int *line_k = nullptr;       // [nl] k1 | plane << 16
    const int *line_row = nullptr;     // [nl + 1] first row
    // work items of a line (ibzk): (row, up to RANKS consecutive in-window ranks)
    const int *line_item = nullptr;    // [nl + 1]
    const int4 *items = nullptr;       // row, k0 | ranks << 8, bands (16 bits each), offset in the output row
    // columns in tiles of CT = 16 ceil(spt nb / 16): column t CT + j nb + i holds
    // inner index i < nb of outer index t spt + j (outer: branch or mp)
    int CT = 16, spt = 1, CPs = 16;
};

constexpr int kAxisMaxCnt = 32;  // cells of one (R0, R1): one thread's chain in stage A (longer ones would run, not measured)
constexpr int kAxisMaxR = 15;    // |R0|, |R1|
constexpr int kAxisMaxN = 62;    // N0, N1

// Band rotation of k_rotate_h (ibzk: h(R) = sum_mp U_k(m, mp) g(k, R)(np, mp, sp) /
// phwsdeg(R)) or branch rotation of k_rotate_hq (ibzq: h(R) = sum_sp u(s, sp)
// g(R, q)(np, mp, sp) / elwsdeg(R)) of the states st0 .. st0 + ns - 1: one wave per
// cell and k (or q), the lanes along the columns; the nrot <= NR values of g are loaded
// once for all states of the k, their coefficients are scalar operands.
struct AxisRotArgs {
    const double2 *g;          // [k][cell][...]
    int64_t g_kstride, cstride;
    int ostride, rstride, nrot;  // elements of g between outer indices and between terms of the rotation
    const int *kst;            // [nk + 1] first state of each k
    const int *st_u;           // coefficient row of a state within its k (ibzk: the band), or null: the state's own
    const double2 *coef;       // [k coef_rows + st_u][nrot], or [state][nrot]
    int coef_rows;
    const int *deg;            // [cell] degeneracy
    int nin, nout;             // inner and outer index counts
    double2 *h;                // [state - st0][entry][CPs]
};
template <int NR>
__global__ __launch_bounds__(256) void k_axis_rot(AxisTab x, AxisRotArgs a, int st0, int ns, int kb0) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e = blockIdx.x * 4 + wave, kb = kb0 + blockIdx.y;
    if (e >= x.ncell) return;
    const sc_int kst = as_scalar(a.kst);
    const int s_lo = max(kst[kb], st0), s_hi = min(kst[kb + 1], st0 + ns);
    const int cell = as_scalar(x.ecell)[e];
    if (cell < 0) {
        for (int st = s_lo; st < s_hi; ++st)
            for (int c = lane; c < x.CPs; c += 64) a.h[((size_t)(st - st0) * x.ncell + e) * x.CPs + c] = make_double2(0.0, 0.0);
        return;
    }
    const double d = 1.0 / (double)as_scalar(a.deg)[cell];
    for (int c = lane; c < x.CPs; c += 64) {
        const int t = c / x.CT, jc = c - t * x.CT, j = jc / a.nin, in = jc - j * a.nin;
        const int outer = t * x.spt + j;
        const bool ok = j < x.spt && outer < a.nout;
        const dv2 *g = reinterpret_cast<const dv2 *>(a.g) + (size_t)kb * a.g_kstride + (size_t)cell * a.cstride +
                       (ok ? (size_t)outer * a.ostride + in : 0);
        dv2 v[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (r < a.nrot) v[r] = g[(size_t)r * a.rstride];
        for (int st = s_lo; st < s_hi; ++st) {
            const sc_dv2 u = as_scalar(a.coef) + (size_t)(a.st_u ? kb * a.coef_rows + as_scalar(a.st_u)[st] : st) * a.nrot;
            double sx = 0.0, sy = 0.0;
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (r < a.nrot) {
                    const dv2 w = u[r];
                    sx = fma(w.x, v[r].x, sx);
                    sx = fma(-w.y, v[r].y, sx);
                    sy = fma(w.x, v[r].y, sy);
                    sy = fma(w.y, v[r].x, sy);
                }
            a.h[((size_t)(st - st0) * x.ncell + e) * x.CPs + c] = ok ? make_double2(sx * d, sy * d) : make_double2(0.0, 0.0);
        }
    }
}

// LDS of k_axis_ab (bytes): F1 of 16 columns (and a zero row), the plane's A
// phases, the pair table, the lines of q1 and the pairs' first entries.
__host__ __device__ inline size_t axis_ab_lds(int np, int ncell, int rm, int r1m, int N1) {
    return ((size_t)(np + 1) * 16 + ncell) * 16 + (((size_t)(2 * rm + 1) * (2 * r1m + 1) * 2 + 15) & ~(size_t)15) +
           (size_t)(N1 + np + 1) * 4;
}

// A and B for 16 columns (tile ct) of one state and plane.  A: a thread sums the
// cells of one (R0, R1) of one column, four at a time, the next four (of this pair or its next
// one) already in flight; pairs with as many cells share a wave, and the zero entries that
// fill up the fours spare it every check.  F1 stays in LDS.  B: a wave takes
// +-R0; with E and D the sum and i times the difference of the rows of R0 and -R0, their
// sums and differences over +-R1 are the operands of the four products that give the
// rows F+ and F- of stage C (row R0 and rm + R0 of F2, lines q1 and N1 - q1).  F2 goes past the
// L2, which keeps the states' h for their planes and tiles.  MT: tiles of 16 q1, 4 KS > r1m.
// The write of F2 bounds it (617 cells, 24^3, 1786 states: 10.3 GB in 2.15 ms, the rate of a
// large copy); with F2 through the L2 3.4 ms, with a check per entry instead of the zero entries 3.3
// and 3.6.
template <int MT, int KS>
__global__ __launch_bounds__(256, MT * KS > 2 ? 1 : 3) void k_axis_ab(AxisTab x, const double2 *__restrict__ h, const int *__restrict__ st_shift,
                                                 int st0, int ns, double2 *__restrict__ F2) {
    extern __shared__ double2 smem[];
    // the states' workgroups by XCD (workgroups go to the XCDs in turn), so that an
    // XCD's L2 serves the reads of its states' h by all their planes and tiles
    const int nct = x.CPs >> 4, per = x.npl * nct;
    const int id = blockIdx.x, r8 = id >> 3, stl = r8 / per * 8 + (id & 7), sub = r8 % per;
    if (stl >= ns) return;
    const int pl = x.pl0 + sub / nct, ct = sub % nct, st = st0 + stl;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    double2 *F1 = smem, *ph = smem + (x.np + 1) * 16;
    unsigned short *pidx = reinterpret_cast<unsigned short *>(ph + x.ncell);
    const int w1 = 2 * x.r1m + 1, npx = (2 * x.rm + 1) * w1;
    int *lineq = reinterpret_cast<int *>(pidx + ((npx + 7) & ~7)), *pe = lineq + x.N1;
    int k1 = 0, k2 = 0;
    if (st_shift) {
        k1 = st_shift[3 * st + 1];
        k2 = st_shift[3 * st + 2];
    }
    int q2 = x.pl_k2[pl] - k2;
    q2 += q2 < 0 ? x.N2 : 0;
    const double2 *pa = x.phA + (size_t)q2 * x.ncell;
    for (int i = tid; i < x.ncell; i += 256) ph[i] = pa[i];
    for (int i = tid; i < npx; i += 256) pidx[i] = x.pidx[i];
    for (int i = tid; i <= x.np; i += 256) pe[i] = x.pe[i];
    for (int i = tid; i < x.N1; i += 256) {
        const int k = i + k1;
        lineq[i] = x.line_of[pl * x.N1 + (k >= x.N1 ? k - x.N1 : k)];
    }
    if (tid < 16) F1[x.np * 16 + tid] = make_double2(0.0, 0.0);
    double co[MT][KS], si[MT][KS];  // cos and sin of 2 pi q1 R1 / N1, R1 = 4 ks + lk
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int R = 4 * ks + lk;
            const double2 t = x.T1[((16 * mt + li) * R) % x.N1];
            co[mt][ks] = R <= x.r1m ? t.x : 0.0;
            si[mt][ks] = R <= x.r1m ? t.y : 0.0;
        }
    __syncthreads();
    {
        const int col = tid & 15;
        const dv2 *hs = reinterpret_cast<const dv2 *>(h) + (size_t)stl * x.ncell * x.CPs + ct * 16 + col;
        auto load = [&](int e, dv2 (&v)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = hs[(unsigned)((e + i) * x.CPs)];
        };
        int P = tid >> 4;
        if (P < x.np) {
            int e = pe[P], e1 = pe[P + 1];
            dv2 v[4];
            load(e, v);
            double sx = 0.0, sy = 0.0;
            while (true) {
                const int Pn = e + 4 < e1 ? P : P + 16;
                int en = e + 4, en1 = e1;
                if (Pn != P) {
                    const int Pc = min(Pn, x.np - 1);
                    en = pe[Pc];
                    en1 = pe[Pc + 1];
                }
                dv2 vn[4];
                load(en, vn);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const double2 w = ph[e + i];
                    sx = fma(w.x, v[i].x, sx);
                    sy = fma(w.x, v[i].y, sy);
                    sx = fma(-w.y, v[i].y, sx);
                    sy = fma(w.y, v[i].x, sy);
                }
                if (Pn != P) {
                    F1[P * 16 + col] = make_double2(sx, sy);
                    sx = sy = 0.0;
                    if (Pn >= x.np) break;
                }
                P = Pn;
                e = en;
                e1 = en1;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = vn[i];
            }
        }
    }
    __syncthreads();
    const size_t lstride = (size_t)(2 * x.rm + 1) * x.CPs;
    double2 *F2s = F2 + (size_t)stl * x.nl * lstride + ct * 16 + li;
    auto put = [](double2 *o, dv2 v) { __builtin_nontemporal_store(v, reinterpret_cast<dv2 *>(o)); };
    for (int R = wave; R <= x.rm; R += 4) {
        d4 ecr[MT], eci[MT], esr[MT], esi[MT], dcr[MT], dci[MT], dsr[MT], dsi[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            ecr[mt] = eci[mt] = esr[mt] = esi[mt] = d4{0, 0, 0, 0};
            dcr[mt] = dci[mt] = dsr[mt] = dsi[mt] = d4{0, 0, 0, 0};
        }
        const unsigned short *pp = pidx + (x.rm + R) * w1 + x.r1m, *pm = pidx + (x.rm - R) * w1 + x.r1m;
        double2 a[KS][4];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int R1 = min(4 * ks + lk, x.r1m);
            // (R1 = 0 and R0 = 0 have no opposite: the zero row)
            a[ks][0] = F1[pp[R1] * 16 + li];
            a[ks][1] = F1[(R1 > 0 ? pp[-R1] : x.np) * 16 + li];
            a[ks][2] = F1[(R > 0 ? pm[R1] : x.np) * 16 + li];
            a[ks][3] = F1[(R > 0 && R1 > 0 ? pm[-R1] : x.np) * 16 + li];
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            // E(+-R1) = sum over +-R0, D(+-R1) = i times the difference
            const double2 e0 = make_double2(a[ks][0].x + a[ks][2].x, a[ks][0].y + a[ks][2].y);
            const double2 e1 = make_double2(a[ks][1].x + a[ks][3].x, a[ks][1].y + a[ks][3].y);
            const double2 f0 = make_double2(a[ks][2].y - a[ks][0].y, a[ks][0].x - a[ks][2].x);
            const double2 f1 = make_double2(a[ks][3].y - a[ks][1].y, a[ks][1].x - a[ks][3].x);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                ecr[mt] = mfma_f64(co[mt][ks], e0.x + e1.x, ecr[mt]);
                eci[mt] = mfma_f64(co[mt][ks], e0.y + e1.y, eci[mt]);
                esr[mt] = mfma_f64(si[mt][ks], e1.y - e0.y, esr[mt]);
                esi[mt] = mfma_f64(si[mt][ks], e0.x - e1.x, esi[mt]);
            }
            if (R > 0)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    dcr[mt] = mfma_f64(co[mt][ks], f0.x + f1.x, dcr[mt]);
                    dci[mt] = mfma_f64(co[mt][ks], f0.y + f1.y, dci[mt]);
                    dsr[mt] = mfma_f64(si[mt][ks], f1.y - f0.y, dsr[mt]);
                    dsi[mt] = mfma_f64(si[mt][ks], f0.x - f1.x, dsi[mt]);
                }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = 16 * mt + lk + 4 * r;
                if (2 * q > x.N1) continue;
                const int la = lineq[q], lb = q > 0 && 2 * q < x.N1 ? lineq[x.N1 - q] : -1;
                if (la >= 0) {
                    double2 *o = F2s + (la - x.l0) * lstride;
                    put(o + R * x.CPs, dv2{ecr[mt][r] + esr[mt][r], eci[mt][r] + esi[mt][r]});
                    if (R > 0) put(o + (x.rm + R) * x.CPs, dv2{dcr[mt][r] + dsr[mt][r], dci[mt][r] + dsi[mt][r]});
                }
                if (lb >= 0) {
                    double2 *o = F2s + (lb - x.l0) * lstride;
                    put(o + R * x.CPs, dv2{ecr[mt][r] - esr[mt][r], eci[mt][r] - esi[mt][r]});
                    if (R > 0) put(o + (x.rm + R) * x.CPs, dv2{dcr[mt][r] - dsr[mt][r], dci[mt][r] - dsi[mt][r]});
                }
            }
    }
}

// LDS of a wave of the C kernels (bytes): the Y tile, reused to stage the results of a
// round.  Row stride of the tile: the epilogues read NBM bands from a row's last
// inner index on (zeros past CT), and an odd stride keeps the rows on distinct banks.
__host__ __device__ inline int axis_ystride(int CT, int nbm, int nb) { return (CT + nbm - nb) | 1; }
__host__ __device__ inline size_t axis_wave_bytes(int N0, int ys, int round_vals) {
    const size_t y = (size_t)N0 * ys * 16, o = (size_t)round_vals * 8;
    return ((y > o ? y : o) + 15) & ~(size_t)15;
}
__host__ __device__ inline size_t axis_items_bytes(int N0, int nb, int ranks) {
    return ((size_t)N0 * ((nb + ranks - 1) / ranks) * 2 + 15) & ~(size_t)15;
}

// Stage C of 16 columns of one line (rows q0, FP64 matrix cores) from the rows of
// F2 in registers, into Yc[q0 ys + column].  4 KS > rm; MT tiles of 16 q.
template <int MT, int KS>
struct AxisC {
    double co[MT][KS], si[MT][KS];  // A operands: cos (R = 4 ks + lk) and sin (R = 4 ks + lk + 1)
    dv2 bc[KS], bs[KS];             // B operands: rows R and rm + R of F2
    unsigned oc[KS], os[KS];        // their offsets within a line's F2
    __device__ __forceinline__ void init(const AxisTab &x, int lane) {
        const int li = lane & 15, lk = lane >> 4;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int q = 16 * mt + li, Rc = 4 * ks + lk, Rs = Rc + 1;
                const double c = x.T0[(q * Rc) % x.N0].x, s = x.T0[(q * Rs) % x.N0].y;
                co[mt][ks] = Rc <= x.rm ? c : 0.0;
                si[mt][ks] = Rs <= x.rm ? s : 0.0;
            }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            // rows past rm have zero coefficients: any row of F2 will do
            oc[ks] = (unsigned)(min(4 * ks + lk, x.rm) * x.CPs + li);
            os[ks] = (unsigned)(min(x.rm + 4 * ks + lk + 1, 2 * x.rm) * x.CPs + li);
        }
    }
    __device__ __forceinline__ void load(const double2 *F2l) {
        const dv2 *p = reinterpret_cast<const dv2 *>(F2l);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            bc[ks] = __builtin_nontemporal_load(p + oc[ks]);
            bs[ks] = __builtin_nontemporal_load(p + os[ks]);
        }
    }
    // forms the tile from the loaded operands, then loads those of `next`
    __device__ __forceinline__ void tile(const double2 *next, int ys, int N0, int lane, double2 *Yc) {
        const int li = lane & 15, lk = lane >> 4;
        d4 cr[MT], ci[MT], sr[MT], sm[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) cr[mt] = ci[mt] = sr[mt] = sm[mt] = d4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                cr[mt] = mfma_f64(co[mt][ks], bc[ks].x, cr[mt]);
                ci[mt] = mfma_f64(co[mt][ks], bc[ks].y, ci[mt]);
                sr[mt] = mfma_f64(si[mt][ks], bs[ks].x, sr[mt]);
                sm[mt] = mfma_f64(si[mt][ks], bs[ks].y, sm[mt]);
            }
        load(next);
        Yc += li;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = 16 * mt + lk + 4 * r;
                if (2 * q <= N0) {
                    Yc[q * ys] = make_double2(cr[mt][r] + sr[mt][r], ci[mt][r] + sm[mt][r]);
                    if (q > 0 && 2 * q < N0)
                        Yc[(N0 - q) * ys] = make_double2(cr[mt][r] - sr[mt][r], ci[mt][r] - sm[mt][r]);
                }
            }
    }
};

// The wave's LDS writes complete before its reads (and its reads before the
// next writes): a wave's LDS requests are served in order.
__device__ __forceinline__ void wave_lds_sync() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// Stage C and the ibzk epilogue (rotations and |g|^2 as in ibzk_epilogue_row),
// fused.  A wave takes one line of one IBZ k and the k's in-window states in turn: they
// have the rows, U_k' and u_q in common.  The line's work items are (row, RANKS
// consecutive in-window ranks), one per lane and round.  For every column tile the wave
// forms Y in LDS and each lane adds its item's share, z(sp) = sum_np conj(U_k'(n, np))
// Y(np, sp), g(s) += u_q(s, sp) z(sp), so nothing per sp is held.  Bands run to
// NBM (U_k' rows padded with zeros): a guard per band would put every LDS
// read of Y in a block of its own and expose its latency.
// VREG: an item's U_k' rows stay in registers.  ULDS (nbr = NBRM): u_q of the line's q
// is copied to LDS once for all states of the k, [sp][q0][s].  Loads from memory
// return in order, so a wait for u loaded by the lanes themselves is a wait for the F2 of the
// next tile, issued before it.
struct AxisKArgs {
    const int *kst;            // [nkb + 1] first state of each k
    const int *st_kint, *st_kb, *st_m;
    const int64_t *st_slot;
    const double2 *Vkp;
    const double2 *uT, *ufT;   // u_q transposed, [q][sp][s]: phonon mesh, electron mesh (mesh_ref > 1)
    const double *wT, *wfT;    // [q][s] 1 / (2 omega) in the units of |g|^2 (0 where omega is 0)
    const double2 *lp, *lpf, *Ukb;  // polar terms (null otherwise), as PairArgs
    int nb, nbr, mesh_ref, Nph0, Nph1;
    double *out;
    int64_t nprocs;
};
__host__ __device__ inline size_t axis_u_bytes(int N0, int nbr) { return (size_t)N0 * nbr * nbr * 16; }
template <int NBM, int NBRM, int RANKS, int MT, int KS, bool VREG, bool ULDS>
__global__ __launch_bounds__(256, 2) void k_axis_pair(AxisTab x, AxisKArgs a, const double2 *__restrict__ F2, int st0, int ns,
                                                      int kb0, int nblk, int msplit) {
    extern __shared__ double2 smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int line = ((int)blockIdx.x % nblk) * 4 + wave;
    if (line >= x.nl) return;  // no workgroup barrier follows
    const int kb = kb0 + blockIdx.y;
    const int s_lo = max(a.kst[kb], st0) + (int)blockIdx.x / nblk, s_hi = min(a.kst[kb + 1], st0 + ns);
    if (s_lo >= s_hi) return;
    const int nb = a.nb, nbr = ULDS ? NBRM : a.nbr, N0 = x.N0;
    const int k0 = a.st_kint[3 * s_lo];
    const int lk12 = x.line_k[x.l0 + line];
    int q1 = (lk12 & 0xffff) - a.st_kint[3 * s_lo + 1], q2 = x.pl_k2[lk12 >> 16] - a.st_kint[3 * s_lo + 2];
    q1 += q1 < 0 ? x.N1 : 0;
    q2 += q2 < 0 ? x.N2 : 0;
    const int ys = axis_ystride(x.CT, NBM, nb), npad = ys - x.CT;
    const size_t wb = axis_wave_bytes(N0, ys, 64 * RANKS * nbr);
    char *wbase = reinterpret_cast<char *>(smem) + wave * (wb + (ULDS ? axis_u_bytes(N0, nbr) : 0));
    double2 *Yw = reinterpret_cast<double2 *>(wbase);
    dv2 *Uw = reinterpret_cast<dv2 *>(wbase + wb);
    auto phonon = [&](int q0) {  // phonon row of q, as phonon_code
        if (q0 % a.mesh_ref == 0 && q1 % a.mesh_ref == 0 && q2 % a.mesh_ref == 0)
            return ((q2 / a.mesh_ref) * a.Nph1 + q1 / a.mesh_ref) * a.Nph0 + q0 / a.mesh_ref;
        return -((q2 * x.N1 + q1) * N0 + q0) - 1;
    };
    auto u_of = [&](int code) {
        return reinterpret_cast<const dv2 *>(code >= 0 ? a.uT : a.ufT) + (size_t)(code >= 0 ? code : -code - 1) * nbr * nbr;
    };
    if constexpr (ULDS) {
        for (int i = lane; i < N0 * NBRM * NBRM; i += 64) {
            const int q0 = i / (NBRM * NBRM), j = i - q0 * (NBRM * NBRM), sp = j / NBRM;
            Uw[(sp * N0 + q0) * NBRM + j - sp * NBRM] = u_of(phonon(q0))[j];
        }
    }
    AxisC<MT, KS> sc;
    sc.init(x, lane);
    const int it0 = x.line_item[x.l0 + line], nit = x.line_item[x.l0 + line + 1] - it0;
    const size_t lsz = (size_t)(2 * x.rm + 1) * x.CPs, ssz = (size_t)x.nl * lsz;
    const double2 *F2l = F2 + (size_t)line * lsz;
    constexpr bool PF = !ULDS && NBRM <= 12;  // u of the next sp loaded ahead
    constexpr int UM = PF ? NBRM : 3, VM = VREG ? NBM : 1;
    for (int i0 = 0; i0 < nit; i0 += 64) {
        // the lane's item
        const bool has = i0 + lane < nit;
        const int4 it = x.items[it0 + min(i0 + lane, nit - 1)];
        const int nr = has ? it.y >> 8 : 0;
        int q0 = (it.y & 0xff) - k0;
        q0 += q0 < 0 ? N0 : 0;
        const int code = phonon(q0);
        const dv2 *uq = ULDS ? Uw + q0 * NBRM : u_of(code);
        const dv2 *V0 = reinterpret_cast<const dv2 *>(a.Vkp) + ((size_t)it.x * nb + (it.z & 0xffff)) * nb;
        const dv2 *V1 = reinterpret_cast<const dv2 *>(a.Vkp) + ((size_t)it.x * nb + (it.z >> 16)) * nb;
        dv2 v[RANKS][VM];
        if constexpr (VREG) {
#pragma unroll
            for (int i = 0; i < NBM; ++i) {
                v[0][i] = i < nb ? V0[i] : dv2{0.0, 0.0};
                if constexpr (RANKS > 1) v[1][i] = i < nb ? V1[i] : dv2{0.0, 0.0};
            }
        }
        const double *w = (code >= 0 ? a.wT : a.wfT) + (size_t)(code >= 0 ? code : -code - 1) * nbr;
        double wr[NBRM];  // (as u: not loaded behind the next F2)
        if constexpr (ULDS)
#pragma unroll
            for (int s = 0; s < NBRM; ++s) wr[s] = w[s];
        const int first = __shfl(it.w, 0), off = it.w - first;
        const int n = __shfl(off + nr * nbr, min(63, nit - i0 - 1));
        sc.load(F2l + (size_t)(s_lo - st0) * ssz);
        for (int st = s_lo; st < s_hi; st += msplit) {
            const double2 *F2c = F2l + (size_t)(st - st0) * ssz;
            const double2 *F2n = st + msplit < s_hi ? F2c + msplit * ssz : F2c;
            dv2 un[UM];
            auto load_u = [&](int sp) {
                const dv2 *up = uq + sp * nbr;
#pragma unroll
                for (int s = 0; s < UM; s += 3)
                    if (s < nbr) {
                        un[s] = up[s];
                        un[s + 1] = up[s + 1];
                        un[s + 2] = up[s + 2];
                    }
            };
            if constexpr (PF) load_u(0);
            double gx[RANKS][NBRM], gy[RANKS][NBRM];
#pragma unroll
            for (int k = 0; k < RANKS; ++k)
#pragma unroll
                for (int s = 0; s < NBRM; ++s) gx[k][s] = gy[k][s] = 0.0;
            // the columns past the tile that the last inner range reads
            for (int i = lane; i < N0 * npad; i += 64) Yw[i / npad * ys + x.CT + i % npad] = make_double2(0.0, 0.0);
            for (int t0 = 0, sp = 0; t0 < x.CPs; t0 += x.CT) {
                for (int cb = 0; cb < x.CT; cb += 16)
                    sc.tile(t0 + cb + 16 < x.CPs ? F2c + t0 + cb + 16 : F2n, ys, N0, lane, Yw + cb);
                wave_lds_sync();
                const double2 *Yr = Yw + q0 * ys;
                for (int j = 0; j < x.spt && sp < nbr; ++j, ++sp, Yr += nb) {
                    double zx[RANKS], zy[RANKS];
#pragma unroll
                    for (int k = 0; k < RANKS; ++k) zx[k] = zy[k] = 0.0;
                    auto mac = [&](int k, dv2 w, double2 y) {  // conj(w) * y
                        zx[k] = fma(w.x, y.x, zx[k]);
                        zy[k] = fma(w.x, y.y, zy[k]);
                        zx[k] = fma(w.y, y.y, zx[k]);
                        zy[k] = fma(-w.y, y.x, zy[k]);
                    };
                    if constexpr (VREG) {
#pragma unroll
                        for (int i = 0; i < NBM; ++i) {
                            const double2 y = Yr[i];
#pragma unroll
                            for (int k = 0; k < RANKS; ++k) mac(k, v[k][i], y);
                        }
                    } else {
#pragma unroll 4
                        for (int i = 0; i < nb; ++i) mac(0, V0[i], Yr[i]);
                    }
                    auto add = [&](int s, dv2 u) {
#pragma unroll
                        for (int k = 0; k < RANKS; ++k) {
                            gx[k][s] = fma(u.x, zx[k], gx[k][s]);
                            gy[k][s] = fma(u.x, zy[k], gy[k][s]);
                            gx[k][s] = fma(-u.y, zy[k], gx[k][s]);
                            gy[k][s] = fma(u.y, zx[k], gy[k][s]);
                        }
                    };
#pragma unroll
                    for (int s = 0; s < NBRM; s += 3)
                        if (s < nbr) {
                            if constexpr (PF) {
                                add(s, un[s]);
                                add(s + 1, un[s + 1]);
                                add(s + 2, un[s + 2]);
                            } else {
                                const dv2 *up = uq + sp * (ULDS ? N0 * NBRM : nbr) + s;
                                const dv2 u0 = up[0], u1 = up[1], u2 = up[2];
                                add(s, u0);
                                add(s + 1, u1);
                                add(s + 2, u2);
                            }
                        }
                    if constexpr (PF) load_u(min(sp + 1, nbr - 1));
                }
                wave_lds_sync();
            }
            // polar term (src/wannier.f90:998-1006)
            if (a.lp) {
                const double2 *lq = (code >= 0 ? a.lp : a.lpf) + (size_t)(code >= 0 ? code : -code - 1) * nbr;
                const double2 *Ukm = a.Ukb + ((size_t)a.st_kb[st] * nb + a.st_m[st]) * nb;
                double2 unm[RANKS];
#pragma unroll
                for (int k = 0; k < RANKS; ++k) {
                    unm[k] = make_double2(0.0, 0.0);
                    const dv2 *V = k ? V1 : V0;
                    for (int i = 0; i < nb; ++i) {
                        const dv2 w = V[i];
                        const double2 t = cmulc(make_double2(w.x, w.y), Ukm[i]);
                        unm[k].x += t.x;
                        unm[k].y += t.y;
                    }
                }
#pragma unroll
                for (int s = 0; s < NBRM; ++s)
                    if (s < nbr) {
                        const double2 l = lq[s];
#pragma unroll
                        for (int k = 0; k < RANKS; ++k) {
                            double2 g = make_double2(gx[k][s], gy[k][s]);
                            cfma(g, l, unm[k]);
                            gx[k][s] = g.x;
                            gy[k][s] = g.y;
                        }
                    }
            }
            // |g|^2 staged over the wave's Y tile (the items' results are one
            // contiguous range of the output), then written by consecutive lanes
            double *stage = reinterpret_cast<double *>(Yw), *o = stage + off;
#pragma unroll
            for (int s = 0; s < NBRM; s += 3)
                if (s < nbr) {
                    double f[3];
#pragma unroll
                    for (int j = 0; j < 3; ++j) f[j] = ULDS ? wr[s + j] : w[s + j];
#pragma unroll
                    for (int k = 0; k < RANKS; ++k)
                        if (k < nr)
#pragma unroll
                            for (int j = 0; j < 3; ++j) {
                                const double x2 = gx[k][s + j] * gx[k][s + j] + gy[k][s + j] * gy[k][s + j];
                                o[k * nbr + s + j] = f[j] != 0.0 ? x2 * f[j] : 0.0;
                            }
                }
            wave_lds_sync();
            double *outrow = a.out + a.st_slot[st] * a.nprocs + first;
            for (int i = lane; i < n; i += 64) __builtin_nontemporal_store(stage[i], outrow + i);
            wave_lds_sync();
        }
    }
}

// Work items of a wave's line: lane r (row r of the line) holds `mine` items,
// listed in row order as row | index << 6; returns their number.
__device__ __forceinline__ int axis_items(int mine, int lane, unsigned short *items) {
    int incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    for (int j = 0; j < mine; ++j) items[incl - mine + j] = (unsigned short)(lane | (j << 6));
    return __builtin_amdgcn_readfirstlane(__shfl(incl, 63));
}

// The same for ibzq (rows k, no shift), the states of one IBZ q in turn: items
// (row, RANKS in-window ranks m); W(np) += U_k(m, mp) Y(np, mp) per column tile
// of mp, then for every in-window n of k' = k + q, g = sum_np conj(U_k'(n, np)) W(np)
// and |g|^2 as in ibzq_row.  Loads return in order: those of U_k for a tile are issued
// ahead of the F2 of the next one, the first U_k'(n) ahead of the next state's, and a lane
// keeps the bands of its k' so that no load waits for another.
template <int NBM, int RANKS, int MT, int KS>
__global__ __launch_bounds__(256, 2) void k_axis_pair_q(AxisTab x, PairQArgs a, const double2 *__restrict__ F2, int st0, int ns,
                                                        int qb0, const int *__restrict__ qst, int nblk, int msplit) {
    extern __shared__ double2 smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int line = ((int)blockIdx.x % nblk) * 4 + wave;
    if (line >= x.nl) return;  // no workgroup barrier follows
    const int qb = qb0 + blockIdx.y;
    const int s_lo = max(qst[qb], st0) + (int)blockIdx.x / nblk, s_hi = min(qst[qb + 1], st0 + ns);
    if (s_lo >= s_hi) return;
    const int nb = a.nb, N0 = x.N0;
    const int ys = axis_ystride(x.CT, NBM, nb), npad = ys - x.CT;
    const size_t wb = axis_wave_bytes(N0, ys, 64 * RANKS * nb), ib = axis_items_bytes(N0, nb, RANKS);
    char *wbase = reinterpret_cast<char *>(smem) + wave * (wb + ib);
    double2 *Yw = reinterpret_cast<double2 *>(wbase);
    unsigned short *items = reinterpret_cast<unsigned short *>(wbase + wb);
    AxisC<MT, KS> sc;
    sc.init(x, lane);
    const int *rowmap = a.rowmap + (size_t)qb * a.nwv;  // (one row set per q)
    const int64_t *rowoff = a.rowoff + (size_t)qb * a.nwv;
    const int row0 = x.line_row[x.l0 + line], nrow = x.line_row[x.l0 + line + 1] - row0;
    int mine = 0;
    if (lane < nrow) {
        const int kp = rowmap[row0 + lane];
        if (kp >= 0 && a.nwin[kp] > 0) mine = (a.nwin[row0 + lane] + RANKS - 1) / RANKS;
    }
    const int nit = axis_items(mine, lane, items);
    wave_lds_sync();
    const size_t lsz = (size_t)(2 * x.rm + 1) * x.CPs, ssz = (size_t)x.nl * lsz;
    const double2 *F2l = F2 + (size_t)line * lsz;
    const dv2 *Vk = reinterpret_cast<const dv2 *>(a.Vk);
    for (int i0 = 0; i0 < nit; i0 += 64) {
        const bool has = i0 + lane < nit;
        const int it = items[min(i0 + lane, nit - 1)], rank = (it >> 6) * RANKS, row = row0 + (it & 63);
        const int nr = has ? min(RANKS, a.nwin[row] - rank) : 0;
        const int yrow = a.kint[3 * row], kp = rowmap[row], nn = a.nwin[kp];
        const int64_t off64 = rowoff[row] + (int64_t)rank * nn;
        const int64_t first = __shfl(off64, 0);
        const int off = (int)(off64 - first), n = __shfl(off + nr * nn, min(63, nit - i0 - 1));
        const dv2 *U[RANKS];
#pragma unroll
        for (int k = 0; k < RANKS; ++k) U[k] = Vk + ((size_t)row * nb + a.wband[row * nb + rank + (k < nr ? k : 0)]) * nb;
        unsigned long long bands = 0;  // in-window bands of k'
        if constexpr (NBM <= 16)
            for (int j = 0; j < nn; ++j) bands |= (unsigned long long)a.wband[kp * nb + j] << (4 * j);
        auto kprow = [&](int nj) {
            return Vk + ((size_t)kp * nb + (NBM <= 16 ? (int)(bands >> (4 * nj)) & 15 : a.wband[kp * nb + nj])) * nb;
        };
        constexpr bool PV = NBM <= 12 && MT * KS <= 2;  // the next n's U_k' loaded ahead (registers)
        dv2 vn[PV ? NBM : 1];
        auto load_v = [&](int nj) {
            const dv2 *v = kprow(nj);
            if constexpr (PV)
#pragma unroll
                for (int i = 0; i < NBM; ++i) vn[i] = i < nb ? v[i] : dv2{0.0, 0.0};
        };
        sc.load(F2l + (size_t)(s_lo - st0) * ssz);
        for (int st = s_lo; st < s_hi; st += msplit) {
            const double2 *F2c = F2l + (size_t)(st - st0) * ssz;
            const double2 *F2n = st + msplit < s_hi ? F2c + msplit * ssz : F2c;
            const double om = a.st_om[st], f = om != 0.0 ? 0.5 * kG2Unit / om : 0.0;
            double Wx[RANKS][NBM], Wy[RANKS][NBM];
#pragma unroll
            for (int k = 0; k < RANKS; ++k)
#pragma unroll
                for (int i = 0; i < NBM; ++i) Wx[k][i] = Wy[k][i] = 0.0;
            dv2 u[2][RANKS];
            auto load_u = [&](int mp) {
#pragma unroll
                for (int k = 0; k < RANKS; ++k) {
                    u[0][k] = U[k][min(mp, nb - 1)];
                    u[1][k] = U[k][min(mp + 1, nb - 1)];
                }
            };
            for (int i = lane; i < N0 * npad; i += 64) Yw[i / npad * ys + x.CT + i % npad] = make_double2(0.0, 0.0);
            for (int t0 = 0, mp = 0; t0 < x.CPs; t0 += x.CT) {
                load_u(mp);
                if (t0 + x.CT >= x.CPs) load_v(0);
                for (int cb = 0; cb < x.CT; cb += 16)
                    sc.tile(t0 + cb + 16 < x.CPs ? F2c + t0 + cb + 16 : F2n, ys, N0, lane, Yw + cb);
                wave_lds_sync();
                const double2 *Yr = Yw + yrow * ys;
                auto mac = [&](int h) {
#pragma unroll
                    for (int i = 0; i < NBM; ++i) {
                        const double2 y = Yr[i];
#pragma unroll
                        for (int k = 0; k < RANKS; ++k) {
                            Wx[k][i] = fma(u[h][k].x, y.x, Wx[k][i]);
                            Wy[k][i] = fma(u[h][k].x, y.y, Wy[k][i]);
                            Wx[k][i] = fma(-u[h][k].y, y.y, Wx[k][i]);
                            Wy[k][i] = fma(u[h][k].y, y.x, Wy[k][i]);
                        }
                    }
                    ++mp;
                    Yr += nb;
                };
                const int m1 = min(mp + x.spt, nb);
                while (mp < m1) {
                    mac(0);
                    if (mp < m1) mac(1);
                    if (mp < m1) load_u(mp);
                }
                wave_lds_sync();
            }
            double *stage = reinterpret_cast<double *>(Yw), *o = stage + off;
            for (int nj = 0; nj < nn; ++nj) {
                const dv2 *Ukp = kprow(nj);
                double2 g[RANKS];
#pragma unroll
                for (int k = 0; k < RANKS; ++k) g[k] = make_double2(0.0, 0.0);
                dv2 v[NBM];
#pragma unroll
                for (int i = 0; i < NBM; ++i)
                    if constexpr (PV) v[i] = vn[i];
                    else v[i] = i < nb ? Ukp[i] : dv2{0.0, 0.0};
                if constexpr (PV) load_v(min(nj + 1, nn - 1));
#pragma unroll
                for (int i = 0; i < NBM; ++i)
#pragma unroll
                    for (int k = 0; k < RANKS; ++k) {
                        g[k].x = fma(v[i].x, Wx[k][i], g[k].x);
                        g[k].y = fma(v[i].x, Wy[k][i], g[k].y);
                        g[k].x = fma(v[i].y, Wy[k][i], g[k].x);
                        g[k].y = fma(-v[i].y, Wx[k][i], g[k].y);
                    }
                if (a.st_lp) {  // src/wannier.f90:998-1006
                    double2 ov[RANKS];
#pragma unroll
                    for (int k = 0; k < RANKS; ++k) ov[k] = make_double2(0.0, 0.0);
                    for (int i = 0; i < nb; ++i) {
                        const dv2 vi = Ukp[i];
#pragma unroll
                        for (int k = 0; k < RANKS; ++k) {
                            const dv2 w = U[k][i];
                            const double2 z = cmulc(make_double2(vi.x, vi.y), make_double2(w.x, w.y));
                            ov[k].x += z.x;
                            ov[k].y += z.y;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < RANKS; ++k) cfma(g[k], a.st_lp[st], ov[k]);
                }
#pragma unroll
                for (int k = 0; k < RANKS; ++k)
                    if (k < nr) o[k * nn + nj] = f != 0.0 ? (g[k].x * g[k].x + g[k].y * g[k].y) * f : 0.0;
            }
            wave_lds_sync();
            double *outrow = a.out + a.st_slot[st] * a.stride + first;
            for (int i = lane; i < n; i += 64) __builtin_nontemporal_store(stage[i], outrow + i);
            wave_lds_sync();
        }
    }
}

// The same three sums at a list of mesh points, for the mixed representations
// g(k, Rp) (cells Re) and g(Re, q) (cells Rp):
//   out[point][column] = sum_R e^{i 2 pi k.R} gwann(R, column) / deg(R).
// Irreducible points lie in few planes and lines (413 of 24^3: 7 planes, 49 lines),
// so the sums over R2 and R1 are shared by many points: 5.9e4 multiply-adds per
// column instead of 5.1e5 of the cell-pair product, which leaves the reads of gwann and the
// writes as the larger part.  A workgroup takes 4 columns (64 bytes of a cell) of one outer
// index: A for up to 8 planes at once (each cell is loaded once for all of them) into
// LDS, then a lane takes one line and column, F2 of all R0 in registers (rows R0 = r - RM,
// RM >= rm), and sums its line's points in the symmetric form.
// Measured for 413 points, 617 cells, 237e3 columns (2.3 GB read, 1.6 GB written): 2.6 ms against
// 10.0 ms in 7 passes of k_gkRp and 6.9 ms in 4 of k_gReq.  Its LDS reads and FP64 operations
// bound it (without the stores 2.4 ms, without the reads beyond L2 2.5); A's phases as scalar
// operands instead of from LDS were slower where few planes are taken (0.54 against 0.23 ms at
// 48 points, 279 cells): every scalar load waits for all of a wave's.
constexpr int kPtsPlanes = 8;
struct AxisCellTab {
    int N0 = 1, N1 = 1, N2 = 1;
    int np = 0, ncell = 0, rm = 0, r1m = 0, r2n = 0;  // pairs, entries, largest |R0|, |R1|, distinct R2
    const int *pe = nullptr;       // [np + 1] first entry of a pair (R0, R1)
    const int *ent = nullptr;      // [ncell] cell | index of its R2 << 16
    const double *dinv = nullptr;  // [ncell] 1 / degeneracy
    const int *poff = nullptr;     // [2 r1m + 1][2 RM + 2] pair of (R0 = r - RM, R1), np where there is none
    const double2 *T0 = nullptr, *T1 = nullptr;  // roots of unity
};
struct AxisPtsArgs {
    const double2 *g;
    int64_t cstride, ostride;  // elements between cells, and between outer indices
    int no, nb2;               // outer indices, contiguous inner columns
    int od;                    // output offset of outer index o: nb2 ((o / od) om + (o % od) on)
    int64_t om, on;
    double2 *out;
    int64_t kstride;           // elements between points
    int npl, nk;
    const int *pl_line;        // [npl + 1] first line of a plane
    const double2 *phA;        // [planes / 8][r2n][8] e^{i 2 pi k2 R2 / N2}
    const int4 *lines;         // k1, first point, points, plane
    const int *ks;             // [nk] points by line: k0 | position in the output << 8
};
__host__ __device__ inline size_t axis_pts_lds(int np, int ncell, int r2n, int N0, int N1, int npl, int nk) {
    const int pl = npl < kPtsPlanes ? npl : kPtsPlanes;
    return ((size_t)pl * (np + 1) * 4 + (size_t)r2n * kPtsPlanes + N0 + N1) * 16 + (size_t)ncell * 12 + (size_t)nk * 4 + 16;
}
template <int RM>
__global__ __launch_bounds__(256, 2) void k_axis_pts(AxisCellTab c, AxisPtsArgs a, int nq) {
    extern __shared__ double2 smem[];
    // nq workgroups share the column tiles of an outer index, all on one XCD; at any time
    // they are at neighbouring tiles, which share cache lines
    const int nt = (a.nb2 + 3) >> 2, id = blockIdx.x, seq = id >> 3;
    const int o = seq / nq * 8 + (id & 7), t0 = seq % nq, t1 = nt;
    if (o >= a.no || t0 >= t1) return;
    const int tid = threadIdx.x, col = tid & 3, slot = tid >> 2;
    const int npl8 = min(a.npl, kPtsPlanes), prow = (c.np + 1) * 4;
    double2 *F1 = smem, *ph2 = F1 + npl8 * prow, *T0s = ph2 + c.r2n * kPtsPlanes, *T1s = T0s + c.N0;
    double *dinv = reinterpret_cast<double *>(T1s + c.N1);
    int *ent = reinterpret_cast<int *>(dinv + c.ncell), *ks = ent + c.ncell;
    for (int i = tid; i < c.N0; i += 256) T0s[i] = c.T0[i];
    for (int i = tid; i < c.N1; i += 256) T1s[i] = c.T1[i];
    for (int i = tid; i < c.ncell; i += 256) {
        ent[i] = c.ent[i];
        dinv[i] = c.dinv[i];
    }
    for (int i = tid; i < a.nk; i += 256) ks[i] = a.ks[i];
    for (int i = tid; i < npl8 * 4; i += 256) F1[(i >> 2) * prow + c.np * 4 + (i & 3)] = make_double2(0.0, 0.0);
    const dv2 *go = reinterpret_cast<const dv2 *>(a.g) + (size_t)o * a.ostride;
    double2 *out = a.out + (size_t)a.nb2 * ((size_t)(o / a.od) * a.om + (size_t)(o % a.od) * a.on);
    const int w1 = 2 * c.r1m + 1;
    for (int p0 = 0; p0 < a.npl; p0 += kPtsPlanes) {
        const int npl = min(kPtsPlanes, a.npl - p0);
        const double2 *ph = a.phA + (size_t)(p0 / kPtsPlanes) * c.r2n * kPtsPlanes;
        for (int i = tid; i < c.r2n * kPtsPlanes; i += 256) ph2[i] = ph[i];
        const int l0 = a.pl_line[p0], l1 = a.pl_line[p0 + npl];
        for (int tile = t0; tile < t1; tile += nq) {
            __syncthreads();  // the tables are there; every wave has read the last tile's F1
            const dv2 *gs = go + min(tile * 4 + col, a.nb2 - 1);
            for (int P = slot; P < c.np; P += 64) {
                const int e0 = c.pe[P], e1 = c.pe[P + 1];
                double sx[kPtsPlanes], sy[kPtsPlanes];
#pragma unroll
                for (int j = 0; j < kPtsPlanes; ++j) sx[j] = sy[j] = 0.0;
                for (int e = e0; e < e1; e += 8) {
                    dv2 v[8];
                    int w[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        w[i] = ent[min(e + i, e1 - 1)];
                        v[i] = gs[(size_t)(w[i] & 0xffff) * a.cstride];
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (e + i < e1) {
                            const double d = dinv[e + i], x = v[i].x * d, y = v[i].y * d;
                            const double2 *t = ph2 + (w[i] >> 16) * kPtsPlanes;
#pragma unroll
                            for (int j = 0; j < kPtsPlanes; ++j) {
                                const double2 u = t[j];
                                sx[j] = fma(u.x, x, sx[j]);
                                sy[j] = fma(u.x, y, sy[j]);
                                sx[j] = fma(-u.y, y, sx[j]);
                                sy[j] = fma(u.y, x, sy[j]);
                            }
                        }
                }
#pragma unroll
                for (int j = 0; j < kPtsPlanes; ++j)
                    if (j < npl) F1[j * prow + P * 4 + col] = make_double2(sx[j], sy[j]);
            }
            __syncthreads();
            const bool colok = tile * 4 + col < a.nb2;
            for (int l = l0 + slot; l < l1; l += 64) {
                const int4 ln = a.lines[l];
                const double2 *f = F1 + (ln.w - p0) * prow + col;
                double ax[2 * RM + 1], ay[2 * RM + 1];
#pragma unroll
                for (int r = 0; r <= 2 * RM; ++r) ax[r] = ay[r] = 0.0;
                int x1 = c.N1 - (c.r1m * ln.x) % c.N1;  // (k1 R1) mod N1 from R1 = -r1m
                x1 = x1 == c.N1 ? 0 : x1;
                for (int i1 = 0; i1 < w1; ++i1) {
                    const double2 w = T1s[x1];
                    x1 += ln.x;
                    x1 -= x1 >= c.N1 ? c.N1 : 0;
                    const sc_int po = as_scalar(c.poff) + i1 * (2 * RM + 2);
#pragma unroll
                    for (int r = 0; r <= 2 * RM; ++r) {
                        const double2 u = f[po[r] * 4];
                        ax[r] = fma(w.x, u.x, ax[r]);
                        ay[r] = fma(w.x, u.y, ay[r]);
                        ax[r] = fma(-w.y, u.y, ax[r]);
                        ay[r] = fma(w.y, u.x, ay[r]);
                    }
                }
                // the symmetric form over R0: sums and i times the differences of +-R0
                double px[RM + 1], py[RM + 1], mx[RM + 1], my[RM + 1];
                px[0] = ax[RM];
                py[0] = ay[RM];
                mx[0] = my[0] = 0.0;
#pragma unroll
                for (int R = 1; R <= RM; ++R) {
                    px[R] = ax[RM + R] + ax[RM - R];
                    py[R] = ay[RM + R] + ay[RM - R];
                    mx[R] = ay[RM - R] - ay[RM + R];
                    my[R] = ax[RM + R] - ax[RM - R];
                }
                double2 *ol = out + tile * 4 + col;
                for (int j = 0; j < ln.z; ++j) {
                    const int k = ks[ln.y + j], k0 = k & 0xff;
                    int x0 = 0;
                    double sx = 0.0, sy = 0.0;
#pragma unroll
                    for (int R = 0; R <= RM; ++R) {
                        const double2 w = T0s[x0];
                        x0 += k0;
                        x0 -= x0 >= c.N0 ? c.N0 : 0;
                        sx = fma(w.x, px[R], sx);
                        sy = fma(w.x, py[R], sy);
                        sx = fma(w.y, mx[R], sx);
                        sy = fma(w.y, my[R], sy);
                    }
                    if (colok) ol[(size_t)(k >> 8) * a.kstride] = make_double2(sx, sy);
                }
            }
        }
        __syncthreads();  // F1 is written again
    }
}
