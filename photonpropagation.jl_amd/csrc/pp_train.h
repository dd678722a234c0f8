// pp_train.h - one training step of the surrogate network in two launches
// (included by pp_mlp.hip, inside its anonymous namespace, after the loss
// head and the fused inference kernel's constants).
//
// A step is small (batch 4096 of the 8-256x4-10 network: 5 GFLOP, 0.8 MB of
// weights), so it is bound by its launches and by the latency of each, not by
// the matrix cores: as one kernel per product, reduction and update it took
// 33 launches and 347 us. Everything that only needs one row of the batch -
// drawing the sample, the forward pass, the loss and the data gradients of
// every layer - is row-local and runs in train_rows_kernel; everything that
// sums over the batch - weight and bias gradients and the Adam update they
// feed - runs in train_grads_kernel. Only the bf16 operands of the weight
// gradients pass through memory between the two (17 MB at batch 4096, in the
// caches); activations stay in LDS, pre-activations in registers, of which they
// leave too few from four hidden layers on: the rows kernel then spills (104 bytes
// of scratch a lane at four, 248 at five, 376 at six; steps of 55, 73 and 88 us at
// batch 4096 against 360, 422 and 489 layer by layer).
//
// Every number is the one the layer-by-layer kernels give: the same 16-term
// MFMA products in the same K order from the same accumulator inputs, the same
// slices of the batch summed in the same order, the same epilogues, and the
// loss's sums over the bins taken bin by bin.

constexpr int kTMaxHidden = 6;  // hidden layers the rows kernel is built for

// Row operands of the weight gradients, H (a layer's input) and D (the gradient
// of its pre-activations), are stored as MFMA operands with the batch as K:
// for 32-column tile T and 16-row block r, 64 lanes x 8 bf16 = 1 KB contiguous,
// chunk (T * nrb + r) * 64 + lane holds column 32T + lane%32 of rows
// 16r + (lane/32)*8 + 0..7. Rows beyond the batch are zero.
struct TrainArgs {
    const float* X;  // features: the dataset (sample) or the batch
    const float* L;  // labels, likewise
    int64_t n;       // samples in the dataset
    int rows;        // batch
    int n_in, n_out;
    bool sample;     // draw the batch's samples (gather_kernel's draw), or take row b as b
    uint32_t k0, k1, step;
    const bf16* Wf[kTMaxHidden + 1];  // packed by pack_weights_kernel: W_l
    const bf16* Wb[kTMaxHidden + 1];  // W_l transposed
    const float* b[kTMaxHidden + 1];
    bf16* H[kTMaxHidden + 1];
    bf16* D[kTMaxHidden + 1];
    int64_t nrb;  // 16-row blocks of H and D (even)
    float inv_rows;
    float* loss;
};

// What the bins of one row share for mixture component j.
struct LossComp {
    float la, k, lth, th, klth, lgk, psi;
};

// The columns of `tiles` 32-column tiles of a [32 rows][kFActLd] LDS tile to
// the packed operand `out` (row blocks rb0, rb0 + 1), zero beyond `valid` rows.
// A wave writes 1 KB contiguous per pass; its LDS reads are along a row.
__device__ __forceinline__ void store_operand(const bf16* act, bf16* out, int tiles, int64_t nrb,
                                              int64_t rb0, int valid) {
    for (int p = threadIdx.x; p < tiles * 128; p += kTThreads) {
        const int lane = p & 63, half = (p >> 6) & 1, tile = p >> 7;
        const int col = tile * 32 + (lane & 31), r0 = half * 16 + (lane >> 5) * 8;
        alignas(16) bf16 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            v[j] = r0 + j < valid ? act[(r0 + j) * kFActLd + col] : (bf16)0.0f;
        *reinterpret_cast<uint4*>(out + ((tile * nrb + rb0 + half) * 64 + lane) * 8) =
            *reinterpret_cast<const uint4*>(v);
    }
}

// One workgroup: 32 rows of the batch through the forward pass, the loss and
// the data gradients. Each wave holds its 32 units' weights of a layer in
// registers (16 fragments), loaded from the packed copies in L2 while the
// layer before is computed: the 128 KB per layer and workgroup are what bounds
// the layers (about 1 us each). Row tiles of 32 leave half of the CUs idle at
// batch 4096; 16-row tiles would fill them but stream the weights twice as
// often and need another MFMA shape, whose sums round differently.
template <int NL>
__global__ void __launch_bounds__(kTThreads) train_rows_kernel(TrainArgs a) {
    __shared__ __attribute__((aligned(16))) bf16 act[2][kTRows * kFActLd];
    __shared__ float lab[kTRows * PP_SUR_LABEL_FLOATS];
    __shared__ float yv[kTRows][33];
    __shared__ LossComp comp[3][kTRows];
    __shared__ float grad[3][3][kTRows];  // sums over the bins: mixture weight, shape, scale
    __shared__ unsigned long long filled[kTRows];  // bins with weight
    __shared__ float bins[7][kTRows * PP_SUR_BINS];  // log p, r[3], x/th[3]
    __shared__ int64_t pick[kTRows];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row0 = blockIdx.x * kTRows;
    const int64_t rb0 = (int64_t)blockIdx.x * 2;
    const int valid = a.rows - row0 < kTRows ? a.rows - row0 : kTRows;
    bf16x8 wn[kFFrag], wc[kFFrag];
    f32x16 z[NL];
    load_weights<2>(a.Wf[0], w, lane, wn);
    if (t < kTRows) {
        int64_t s = -1;
        if (t < valid) {
            s = row0 + t;
            if (a.sample) {
                const uint4 r = pp::philox(make_uint4((uint32_t)s, a.step, 0x5EEDBA7Cu, 0u), a.k0,
                                           a.k1);
                s = (int64_t)__umul64hi(((uint64_t)r.x << 32) | r.y, (uint64_t)a.n);
            }
        }
        pick[t] = s;
    }
    __syncthreads();
    for (int i = t; i < kTRows * 32; i += kTThreads) {
        const int64_t s = pick[i >> 5];
        const int k = i & 31;
        act[0][(i >> 5) * kFActLd + k] =
            s >= 0 && k < a.n_in ? (bf16)a.X[s * a.n_in + k] : (bf16)0.0f;
    }
    for (int i = t; i < kTRows * PP_SUR_LABEL_FLOATS; i += kTThreads) {
        const int64_t s = pick[i / PP_SUR_LABEL_FLOATS];
        lab[i] = s >= 0 ? a.L[s * PP_SUR_LABEL_FLOATS + i % PP_SUR_LABEL_FLOATS] : 0.0f;
    }
    __syncthreads();
    // ---- forward: layer l reads act[l & 1], writes act[(l + 1) & 1]
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const bf16* in = act[l & 1];
        bf16* out = act[(l + 1) & 1];
        f32x16 acc = bias_block(a.b[l], 32 * w, kFH, lane);
#pragma unroll
        for (int i = 0; i < kFFrag; ++i) wc[i] = wn[i];
        if (l + 1 < NL)
            load_weights<kFFrag>(a.Wf[l + 1], w, lane, wn);
        else if (w == 0)
            load_weights<kFFrag>(a.Wf[NL], 0, lane, wn);
        __builtin_amdgcn_sched_barrier(0);
        acc = l == 0 ? tile_product<2>(acc, wc, in, lane) : tile_product<kFFrag>(acc, wc, in, lane);
        z[l] = acc;
        store_silu(acc, out, w, lane);
        store_operand(in, a.H[l], l == 0 ? 1 : kFH / 32, a.nrb, rb0, valid);
        __syncthreads();
    }
    bf16* const top = act[NL & 1];
    if (w == 0) {
        f32x16 acc = bias_block(a.b[NL], 0, a.n_out, lane);
        acc = tile_product<kFFrag>(acc, wn, top, lane);
#pragma unroll
        for (int r = 0; r < 16; ++r)
            yv[lane & 31][(r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)] = acc[r];
    }
    load_weights<2>(a.Wb[NL], w, lane, wn);
    store_operand(top, a.H[NL], kFH / 32, a.nrb, rb0, valid);
    __syncthreads();
    // ---- loss (loss_head_kernel's, a row per group of threads): the mixture's
    // components, then the bins that hold weight, then the sums over them
    if (t < 3 * kTRows) {
        const int j = t / kTRows, r = t % kTRows;
        const float* y = yv[r];
        const float amax = fmaxf(fmaxf(y[1], y[2]), y[3]);
        const float lse = amax + logf(__expf(y[1] - amax) + __expf(y[2] - amax) + __expf(y[3] - amax));
        LossComp c;
        c.la = y[1 + j] - lse;
        c.k = __expf(fminf(fmaxf(y[4 + j], kShapeLo), kShapeHi));
        c.lth = fminf(fmaxf(y[7 + j], kScaleLo), kScaleHi) + 4.0f;
        c.th = __expf(c.lth);
        c.klth = c.k * c.lth;
        c.lgk = lgammaf(c.k);
        c.psi = digamma_f(c.k);
        comp[j][r] = c;
    }
    __syncthreads();
    {
#pragma clang fp contract(off)
        const float x = ((float)lane + 0.5f) * (PP_SUR_TMAX / PP_SUR_BINS), lx = logf(x);
        for (int r = w; r < kTRows; r += kTThreads / 64) {
            const float h = lab[r * PP_SUR_LABEL_FLOATS + 2 + lane];
            const unsigned long long m = __ballot(h != 0.0f);
            if (lane == 0) filled[r] = m;
            if (h != 0.0f) {
                float l[3], xt[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const LossComp c = comp[j][r];
                    xt[j] = x / c.th;
                    l[j] = fmaf(lx, c.k - 1.0f, c.la) - xt[j] - c.klth - c.lgk;
                }
                const float lm = fmaxf(fmaxf(l[0], l[1]), l[2]);
                const float lp =
                    lm + logf(__expf(l[0] - lm) + __expf(l[1] - lm) + __expf(l[2] - lm));
                const int o = r * PP_SUR_BINS + lane;
                bins[0][o] = lp;
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    bins[1 + j][o] = __expf(l[j] - lp);
                    bins[4 + j][o] = xt[j];
                }
            }
        }
        __syncthreads();
        if (t < 3 * kTRows) {
            const int j = t / kTRows, r = t % kTRows;
            const LossComp c = comp[j][r];
            float gl = 0.0f, gs = 0.0f, gc = 0.0f;
            for (unsigned long long m = filled[r]; m; m &= m - 1) {
                const int i = __builtin_ctzll(m), o = r * PP_SUR_BINS + i;
                const float h = lab[r * PP_SUR_LABEL_FLOATS + 2 + i];
                const float p = bins[1 + j][o], xt = bins[4 + j][o];
                const float li = logf(((float)i + 0.5f) * (PP_SUR_TMAX / PP_SUR_BINS));
                const float hp = h * p;
                gl = fmaf(-h, p, gl);
                gs = fmaf(-(li - c.lth - c.psi), c.k * hp, gs);
                gc = fmaf(-(xt - c.k), hp, gc);
            }
            const float ys = yv[r][4 + j], yc = yv[r][7 + j];
            grad[0][j][r] = gl;
            grad[1][j][r] = ys < kShapeLo || ys > kShapeHi ? 0.0f : gs;
            grad[2][j][r] = yc < kScaleLo || yc > kScaleHi ? 0.0f : gc;
        } else if (t < 4 * kTRows) {
            const int r = t % kTRows;
            float lb = 0.0f;
            if (r < valid) {
                const float n_mc = lab[r * PP_SUR_LABEL_FLOATS];
                const float wt = lab[r * PP_SUR_LABEL_FLOATS + 1];
                const float y0 = fminf(fmaxf(yv[r][0], kY0Lo), kY0Hi);
                lb = fmaf(-wt, logf(n_mc) + y0, n_mc * __expf(y0));
                for (unsigned long long m = filled[r]; m; m &= m - 1) {
                    const int i = __builtin_ctzll(m);
                    lb = fmaf(-lab[r * PP_SUR_LABEL_FLOATS + 2 + i], bins[0][r * PP_SUR_BINS + i], lb);
                }
            }
            // the workgroup's loss: the half wave's 32 rows, one atomic
            lb *= a.inv_rows;
            for (int o = 16; o > 0; o >>= 1) lb += __shfl_xor(lb, o);
            if (r == 0) atomicAdd(a.loss, lb);
        }
        __syncthreads();
        bf16* dy = act[(NL + 1) & 1];
        for (int i = t; i < kTRows * 32; i += kTThreads) {
            const int r = i >> 5, o = i & 31;
            float g = 0.0f;
            if (r < valid && o < PP_SUR_N_OUT) {
                if (o == 0) {
                    const float n_mc = lab[r * PP_SUR_LABEL_FLOATS];
                    const float wt = lab[r * PP_SUR_LABEL_FLOATS + 1];
                    const float y0 = fminf(fmaxf(yv[r][0], kY0Lo), kY0Hi);
                    g = yv[r][0] >= kY0Lo && yv[r][0] <= kY0Hi ? n_mc * __expf(y0) - wt : 0.0f;
                } else if (o < 4) {
                    const float sum = grad[0][0][r] + grad[0][1][r] + grad[0][2][r];
                    g = fmaf(-__expf(comp[o - 1][r].la), sum, grad[0][o - 1][r]);
                } else {
                    g = o < 7 ? grad[1][o - 4][r] : grad[2][o - 7][r];
                }
            }
            dy[r * kFActLd + o] = (bf16)(g * a.inv_rows);
        }
        __syncthreads();
    }
    // ---- data gradients: matrix l takes act[(l + 1) & 1] to act[l & 1]
#pragma unroll
    for (int l = NL; l >= 1; --l) {
        const bf16* in = act[(l + 1) & 1];
        bf16* out = act[l & 1];
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < kFFrag; ++i) wc[i] = wn[i];
        if (l > 1) load_weights<kFFrag>(a.Wb[l - 1], w, lane, wn);
        __builtin_amdgcn_sched_barrier(0);
        acc = l == NL ? tile_product<2>(acc, wc, in, lane) : tile_product<kFFrag>(acc, wc, in, lane);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            bf16 d[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float zz = z[l - 1][4 * g + j], s = sigmoid(zz);
                d[j] = (bf16)(acc[4 * g + j] * (s * (1.0f + zz * (1.0f - s))));
            }
            *reinterpret_cast<uint2*>(out + (lane & 31) * kFActLd + 32 * w + 8 * g +
                                      (lane >> 5) * 4) = *reinterpret_cast<const uint2*>(d);
        }
        store_operand(in, a.D[l], l == NL ? 1 : kFH / 32, a.nrb, rb0, valid);
        __syncthreads();
    }
    store_operand(act[1], a.D[0], kFH / 32, a.nrb, rb0, valid);
}

// Parameters after one Adam(W) step: adam_kernel's arithmetic, with the bias
// corrections 1 - beta^t passed in.
__device__ __forceinline__ float adam_update(const pp_adam& o, float g, float c1, float c2, float& m,
                                             float& v, float p) {
#pragma clang fp contract(off)
    m = fmaf(1.0f - o.beta1, g, o.beta1 * m);
    v = fmaf(g, (1.0f - o.beta2) * g, o.beta2 * v);
    const float mh = m / c1, vh = v / c2;
    return fmaf(-o.lr, fmaf(o.weight_decay, p, mh / (sqrtf(vh) + o.eps)), p);
}

struct GradLayer {
    const bf16 *H, *D;
    bf16 *Wf, *Wb;        // packed copies that the update refreshes
    int64_t w_off, b_off;
    int n_i, n_o;
    int k_chunk, slices;  // batch rows per slice of the weight gradient, slices
    int tiles_i;          // 32-wide tiles of the inputs
    int first_w, first_b; // first workgroup of the weight tiles, of the bias tiles
};

struct GradArgs {
    GradLayer layer[kTMaxHidden + 1];
    int n_mat;
    int rows;
    int64_t nrb;
    bool update;  // Adam and the packed copies; otherwise the gradients alone
    float* g;
    float *p, *m, *v;
    bf16* pb;
    pp_adam o;
    uint32_t step;  // steps taken before this one
};

// Weight and bias gradients of every layer in one launch, the sums over the
// batch finished inside the workgroup, and (update) the Adam step of the same
// parameters with the refreshed bf16 copies: no partial sums in memory, no
// gradient round trip, no separate reductions, update and packing.
// A workgroup takes one 32 x 32 tile of a weight matrix (208 of them for the
// 8-256x4-10 network, about one per CU); its eight waves take the batch's
// slices in turn and the slices' products are added in ascending order, as
// reduce_partials_kernel adds them. Bound by the operand reads from L2 (2 KB
// per product; 512 KB per workgroup at batch 4096).
__global__ void __launch_bounds__(kTThreads) train_grads_kernel(GradArgs a) {
    __shared__ float red[8][32 * 32];
    __shared__ bf16 packed[32][36];
    __shared__ float corr[2];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int blk = blockIdx.x;
    if (a.update && t == 0) {
        const float st = (float)(a.step + 1);
        corr[0] = 1.0f - powf(a.o.beta1, st);
        corr[1] = 1.0f - powf(a.o.beta2, st);
    }
    // the weight tiles of every layer, then their bias tiles
    const bool bias = blk >= a.layer[0].first_b;
    int l = 0;
    for (int i = 1; i < a.n_mat; ++i)
        if (blk >= (bias ? a.layer[i].first_b : a.layer[i].first_w)) l = i;
    const GradLayer& q = a.layer[l];
    if (bias) {
        // column sums of D: 64-row chunks, each as four interleaved sums
        // (colsum_kernel), added in ascending order
        const int tile = blk - q.first_b, col = t & 31;
        const int chunks = (a.rows + 63) / 64;
        float total = 0.0f;
        for (int c0 = 0; c0 < chunks; c0 += 16) {
            const int c = c0 + (t >> 5);
            float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (c < chunks) {
                for (int k = 0; k < 8; ++k) {
                    const int64_t rb = (int64_t)c * 4 + (k >> 1);
                    if (rb >= a.nrb) break;
                    const bf16x8 d = *reinterpret_cast<const bf16x8*>(
                        q.D + ((tile * a.nrb + rb) * 64 + col + 32 * (k & 1)) * 8);
#pragma unroll
                    for (int j = 0; j < 8; ++j) s[j & 3] += (float)d[j];
                }
            }
            red[0][t] = (s[0] + s[1]) + (s[2] + s[3]);
            __syncthreads();
            if (t < 32)
                for (int k = 0; k < 16 && c0 + k < chunks; ++k) total += red[0][32 * k + t];
            __syncthreads();
        }
        const int u = tile * 32 + t;
        if (t < 32 && u < q.n_o) {
            const int64_t i = q.b_off + u;
            if (!a.update) {
                a.g[i] = total;
            } else {
                float m = a.m[i], v = a.v[i];
                const float p = adam_update(a.o, total, corr[0], corr[1], m, v, a.p[i]);
                a.m[i] = m;
                a.v[i] = v;
                a.p[i] = p;
                a.pb[i] = (bf16)p;
            }
        }
        return;
    }
    const int tile = blk - q.first_w, to = tile / q.tiles_i, ti = tile % q.tiles_i;
    const bf16x8* A = reinterpret_cast<const bf16x8*>(q.D) + (to * a.nrb) * 64 + lane;
    const bf16x8* B = reinterpret_cast<const bf16x8*>(q.H) + (ti * a.nrb) * 64 + lane;
    float total[2] = {0.0f, 0.0f};
    for (int s0 = 0; s0 < q.slices; s0 += 8) {
        const int s = s0 + w;
        if (s < q.slices) {
            f32x16 acc;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
            const int64_t b0 = (int64_t)s * q.k_chunk / 16;
            const int64_t b1 = b0 + q.k_chunk / 16 < a.nrb ? b0 + q.k_chunk / 16 : a.nrb;
            int64_t b = b0;
            for (; b + 8 <= b1; b += 8) {
                bf16x8 fa[8], fb[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    fa[i] = A[(b + i) * 64];
                    fb[i] = B[(b + i) * 64];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[i], acc, 0, 0, 0);
            }
            for (; b < b1; ++b)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[b * 64], B[b * 64], acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                red[w][((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * 32 + (lane & 31)] = acc[r];
        }
        __syncthreads();
        const int k1 = q.slices - s0 < 8 ? q.slices - s0 : 8;
        for (int k = 0; k < k1; ++k) {
            total[0] += red[k][t];
            total[1] += red[k][t + kTThreads];
        }
        __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int m32 = (t + e * kTThreads) >> 5, n32 = t & 31;
        const int o = to * 32 + m32, in = ti * 32 + n32;
        bf16 pb = (bf16)0.0f;
        if (o < q.n_o && in < q.n_i) {
            const int64_t i = q.w_off + (int64_t)o * q.n_i + in;
            if (!a.update) {
                a.g[i] = total[e];
            } else {
                float m = a.m[i], v = a.v[i];
                const float p = adam_update(a.o, total[e], corr[0], corr[1], m, v, a.p[i]);
                a.m[i] = m;
                a.v[i] = v;
                a.p[i] = p;
                pb = (bf16)p;
                a.pb[i] = pb;
            }
        }
        packed[m32][n32] = pb;
    }
    if (!a.update) return;
    __syncthreads();
    // the tile's two fragments in each packed copy, 2 KB contiguous each
    if (t < 256) {
        const int f = (t >> 6) & 1, c = lane & 31, k0 = 16 * f + (lane >> 5) * 8;
        alignas(16) bf16 v[8];
        const bool fwd = t < 128;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = fwd ? packed[c][k0 + j] : packed[k0 + j][c];
        const int64_t nf = fwd ? 2 * q.tiles_i : (q.n_o + 31) / 32 * 2;
        const int64_t chunk = (fwd ? to * nf + 2 * ti : ti * nf + 2 * to) + f;
        bf16* out = fwd ? q.Wf : q.Wb;
        if (out)
            *reinterpret_cast<uint4*>(out + (chunk * 64 + lane) * 8) =
                *reinterpret_cast<const uint4*>(v);
    }
}
