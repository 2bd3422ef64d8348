// Whole paths in one launch for scenes with unbounded SDF objects (included by kernels.hip inside its anonymous
// namespace, after trace.hpp).
//
// A launch of k_march per depth ends with its longest march -- a grazing ray takes 256 Mandelbulb steps, half a
// millisecond on its own -- so a frame waited for one such march per depth.  Here a lane holds a path and takes it
// from vertex to vertex: the closest bounded hit, the march of each unbounded object in list order with the closest
// hit so far as its cut, the six estimates of an SDF hit's normal, and the shading, while the other lanes are at
// theirs.  Marches and normals are both "the estimate of SDF j at a point", so every pass of the wave evaluates one
// SDF for all the lanes that are at it: the SDF most lanes want, read at a wave-uniform address; the lanes at another
// one wait until theirs is.  Hits are shaded, lanes without a path take new ones, and new rays are traced through the
// bounded objects' tree once enough lanes wait for that.
//
// Each march is k_march's (the same steps, exits and outcomes), each normal sdf_normal's, and the merge's order is
// kept: object by object, strict < against the closest hit so far.  Bound by VALU issue (1.366 wave64 instructions per
// CU per cycle, 45.2% of lanes active, on the 720p frame) and, for small frames, by the serial chain of the longest
// path's estimates.  Per call, before and after: the 161x91, 9-sample SDF frame 8.9 -> 4.4 ms, the 720p, 128-sample
// one 76.1 -> 66 (launched_depths says which depths stay apart), the batch of 16 requests 29.1 -> 20.3.

// Waves per SIMD (the 161x91, 9-sample SDF frame at 4, 5 and 6: 4.6, 4.5 and 4.2 ms, the 64x36, 2-sample one at 5 and
// 6: 3.2 and 3.4, the 720p, 128-sample one 83 and 82), and the lanes that wait before a wave shades, takes new
// paths and traces their rays through the tree: fewer where that is cheap beside a pass of estimates, as it is beside a
// Mandelbulb's iterations, more where it is the work and estimates are cheap.  (At 16, 32 and 48: the Mandelbulb scene
// at 1280x720x128 71.8, 76.0 and above 81 ms, at 640x360x64 17.2, 17.9 and 19.5; a scene of 60 bounded objects and one
// sphere SDF at 1280x720x64 19.0, 14.2 and 13.5 ms, at 333x217x30 3.20, 2.72 and 2.64.  "No Mandelbulb" stands for cheap
// estimates: sixteen smooth-min spheres alone, whose estimates are not, would rather wait for fewer, at 16, 24, 48 and 63
// lanes 12.4, 12.1, 12.8 and 16.0 ms at 1280x720x64 and 4.21, 4.23, 4.61 and 5.35 at 640x360x64; trace_tuning has the
// shares of refill_lanes.)  Once there are no paths left to take, a quarter of its paths (the 161x91, 9-sample frame at
// half, a quarter, an eighth and a sixty-fourth: 4.31, 4.19, 4.20 and 4.28 ms).
constexpr int SDF_TRACE_WAVES = 5;

template <bool BATCH, bool INST, bool SPH, bool VOL, bool TEX, bool ADJOINT>
__global__ __launch_bounds__(EXT_BLOCK) __attribute__((amdgpu_waves_per_eu(SDF_TRACE_WAVES))) void k_trace_sdf(
    TraceArgs args) {
    __shared__ unsigned long long s_entry[EXT_LDS_STACK * EXT_BLOCK];
    __shared__ float s_t[3 * EXT_BLOCK];  // the paths' throughputs
    const GSdf *__restrict__ sdfs = args.sv.sdfs;
    const GSphere *__restrict__ spheres = args.sv.spheres;
    const uint32_t count = args.queue ? *args.count : args.fp.n_slots;
    const uint32_t gid = blockIdx.x * EXT_BLOCK + threadIdx.x;
    const uint32_t lane = __lane_id();
    LaneStack st{(lds_u64 *)s_entry, args.overflow + gid, gridDim.x * EXT_BLOCK, 0};
    enum : int { IDLE, MARCH, NORMAL, HIT };  // no path; marching object j; at an SDF hit's normal; to be shaded
    int state = IDLE;
    uint32_t slot = 0, depth = 0, n_segments = 0;
    DRay ray{};
    Best b{FLT_MAX, -1, 0u, 0u, 0u};  // the closest hit so far
    int32_t j = 0, j_end = 0;         // the SDF marched (or, at the normal, hit) and the end of the scene's SDFs
    float total = 0.0f;               // MARCH: the distance marched; NORMAL: the estimate at +epsilon
    int step = 0;                     // the march's step; the normal's estimate (0..5: +x -x +y -y +z -z)
    f3 g{0.0f, 0.0f, 0.0f};           // the estimate's differences, then the normal
    WaveClaims claims(count, EXT_BLOCK / 64, TRACE_CLAIM_LEAST, args.tune.wave_batch, args.work);
    const uint32_t refill_lanes = args.tune.refill_lanes;
    TravStats stats;
    // the path's RNG key, pixel and sample, and in a batch its request
    auto identify = [&](const TraceArgs &A, dm::Key *key, uint32_t *pixel, uint32_t *sample) -> const RequestParams * {
        if (BATCH) {
            const RequestParams *R = A.bv.reqs + A.bv.slot_req[slot];
            const uint32_t l = slot - R->slot_base;
            *key = dm::Key{R->key0, R->key1};
            *pixel = l / R->n_spp;
            *sample = R->s0 + l % R->n_spp;
            return R;
        }
        *key = dm::Key{A.fp.key0, A.fp.key1};
        *pixel = slot / A.fp.n_spp;
        *sample = A.fp.s0 + slot % A.fp.n_spp;
        return nullptr;
    };
    for (;;) {
        const unsigned long long paths = __ballot(state != IDLE), waiting = __ballot(state == HIT) | ~paths;
        const uint32_t n_idle = 64u - (uint32_t)__popcll(paths), n_hit = (uint32_t)__popcll(waiting) - n_idle;
        if (waiting == ~0ull ||
            (claims.exhausted ? 4u * n_hit >= 64u - n_idle : n_idle + n_hit >= refill_lanes)) {
            const TraceArgs &A = cold_args();
            bool begin = false;
            VertexGrad grad;
            if (state == HIT) {
                dm::Key key;
                uint32_t pixel, sample;
                const RequestParams *R = identify(A, &key, &pixel, &sample);
                const Col T{s_t[threadIdx.x], s_t[EXT_BLOCK + threadIdx.x], s_t[2 * EXT_BLOCK + threadIdx.x]};
                Col L{0.0f, 0.0f, 0.0f}, add{0.0f, 0.0f, 0.0f};
                if (ADJOINT) L = Col{A.pb.lr[slot], A.pb.lg[slot], A.pb.lb[slot]};
                const uint32_t at_depth = depth;
                const Best hit = b;
                begin = shade_vertex<ADJOINT, TEX, false, false>(
                    A.sv, nullptr, A.ap, grad, ray, hit.ref, &hit.t, &hit.aux, &hit.sub, true, g, key, pixel, sample,
                    at_depth, BATCH ? R->ray_depth : A.fp.ray_depth, BATCH ? R->skybox : A.sv.skybox,
                    BATCH ? R->sky_image : A.sv.sky_image, T, L, add, [&](const DRay &nr, const Col &t) {
                        ray.o = nr.o;
                        ray.d = nr.d;
                        s_t[threadIdx.x] = t.r;
                        s_t[EXT_BLOCK + threadIdx.x] = t.g;
                        s_t[2 * EXT_BLOCK + threadIdx.x] = t.b;
                        ++depth;
                    });
                const bool adds = !(add.r == 0.0f && add.g == 0.0f && add.b == 0.0f);
                if (!ADJOINT && at_depth != 0u && adds) L = Col{A.pb.lr[slot], A.pb.lg[slot], A.pb.lb[slot]};
                if (!ADJOINT) L = L + add;
                if (ADJOINT || at_depth == 0u || adds) {
                    A.pb.lr[slot] = L.r;
                    A.pb.lg[slot] = L.g;
                    A.pb.lb[slot] = L.b;
                }
                state = IDLE;
            }
            if (ADJOINT) add_grads(A.ap, blockIdx.x % A.ap.copies, grad);
            const unsigned long long idle = __ballot(state == IDLE && !begin);
            if (!claims.exhausted && idle != 0ull) {
                const uint32_t q = claims.hand_out(idle);
                if (state == IDLE && !begin && q != 0xffffffffu) {
                    slot = A.queue ? (uint32_t)A.queue[q] : q;
                    depth = A.first_depth;
                    Col T{1.0f, 1.0f, 1.0f};
                    if (A.first_depth == 0u) {
                        dm::Key key;
                        uint32_t pixel, sample;
                        const RequestParams *R = identify(A, &key, &pixel, &sample);
                        const DRay c = BATCH ? camera_ray(R->vp, R->width, R->height, R->sdim, key, pixel, sample)
                                             : camera_ray(A.fp.vp, A.fp.width, A.fp.height, A.fp.sdim, key, pixel, sample);
                        ray.o = c.o;
                        ray.d = c.d;
                    } else {
                        ray.o = f3{A.pb.ox[slot], A.pb.oy[slot], A.pb.oz[slot]};
                        ray.d = f3{A.pb.dx[slot], A.pb.dy[slot], A.pb.dz[slot]};
                        T = Col{A.pb.tr[slot], A.pb.tg[slot], A.pb.tb[slot]};
                    }
                    s_t[threadIdx.x] = T.r;
                    s_t[EXT_BLOCK + threadIdx.x] = T.g;
                    s_t[2 * EXT_BLOCK + threadIdx.x] = T.b;
                    begin = true;
                }
            }
            if (begin) {  // the closest bounded hit
                dm::Key key;
                uint32_t pixel, sample;
                const RequestParams *R = identify(A, &key, &pixel, &sample);
                if (INST) {  // finish_instance reloads the world ray
                    A.pb.ox[slot] = ray.o.x;
                    A.pb.oy[slot] = ray.o.y;
                    A.pb.oz[slot] = ray.o.z;
                    A.pb.dx[slot] = ray.d.x;
                    A.pb.dy[slot] = ray.d.y;
                    A.pb.dz[slot] = ray.d.z;
                }
                const int32_t root = BATCH ? R->root : A.sv.root;
                b = Best{FLT_MAX, -1, 0u, 0u, 0u};
                LeafRange leaf;
                st.sp = 0;
                st.top_valid = false;
                if (root >= 0) st.push(root, -__builtin_inff());
                DRay r = ray_from_dir(ray.o, ray.d);
                while (st.sp > 0 || leaf.code != 0)
                    traverse_pass<INST, SPH, VOL>(A.sv, A.pb, slot, r, b, leaf, st, key, pixel, sample, depth, stats);
                j = BATCH ? R->first_sdf : 0;
                j_end = j + (BATCH ? R->n_sdfs : A.sv.n_sdfs);
                total = T_MIN;
                step = 0;
                state = j < j_end ? MARCH : HIT;
                ++n_segments;
            }
        }
        const unsigned long long at_sdf = __ballot(state == MARCH || state == NORMAL);
        if (at_sdf == 0ull) {
            if (claims.exhausted && !__any(state == HIT)) break;
            continue;
        }
        // of the first two SDFs that lanes are at, the one with more of them
        int32_t js = __builtin_amdgcn_readlane(j, __ffsll((long long)at_sdf) - 1);
        unsigned long long at_js = __ballot(j == js) & at_sdf;
        const unsigned long long rest = at_sdf & ~at_js;
        if (rest != 0ull) {
            const int32_t j2 = __builtin_amdgcn_readlane(j, __ffsll((long long)rest) - 1);
            const unsigned long long at_j2 = __ballot(j == j2) & at_sdf;
            if (__popcll(at_j2) > __popcll(at_js)) {
                js = j2;
                at_js = at_j2;
            }
        }
        if (((at_js >> lane) & 1ull) != 0ull) {
            const GSdf &f = sdfs[js];
            const float e = step & 1 ? -f.epsilon : f.epsilon;
            f3 point = at(ray, state == MARCH ? total : b.t);
            if (state == NORMAL) {
                if (step < 2) point.x = point.x + e;
                else if (step < 4) point.y = point.y + e;
                else point.z = point.z + e;
            }
            const f3 qe = point - f3{f.ex, f.ey, f.ez};
            bool ended = state == MARCH &&
                         (total >= b.t || (dot(qe, qe) > f.escape_r * f.escape_r && dot(qe, ray.d) > 0.0f));
            if (!ended) {
                const float dist = sdf_eval(spheres, f, point);
                if (state == MARCH) {
                    total = total + fabsf(dist);
                    if (fabsf(dist) < f.epsilon && T_MIN <= total && total <= FLT_MAX) {
                        if (total < b.t)
                            b = Best{total, -1, make_ref(ITEM_SDF, js),
                                     (signbit(dist) ? HIT_AUX_BACK : 0u) | ((uint32_t)step << HIT_AUX_SIDE_SHIFT), 0u};
                        ended = true;
                    } else {
                        ended = step > f.max_iterations;
                        ++step;
                    }
                } else {
                    if (!(step & 1)) {
                        total = dist;
                    } else {
                        const float d = total - dist;
                        if (step == 1) g.x = d;
                        else if (step == 3) g.y = d;
                        else g.z = d;
                    }
                    if (++step == 6) {
                        g = normalize(g);
                        state = HIT;
                    }
                }
            }
            if (ended) {  // the next unbounded object, or the hit's normal
                total = T_MIN;
                step = 0;
                if (++j == j_end) {
                    const bool sdf_hit = (b.ref >> HIT_KIND_SHIFT) == (uint32_t)ITEM_SDF;
                    if (sdf_hit) j = (int32_t)(b.ref & HIT_INDEX_MASK);
                    state = sdf_hit ? NORMAL : HIT;
                }
            }
        }
    }
    stats.flush();
    add_segments(args.segments, n_segments);
}
