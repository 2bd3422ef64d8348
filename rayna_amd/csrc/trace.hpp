// Whole paths in one launch (included by kernels.hip inside its anonymous namespace, after shade_vertex).
//
// A lane holds a path: it traverses the path's ray (k_extend's loops), and once enough lanes of the wave wait with
// their closest hit or without a path, those hits are shaded, the surviving paths go on with their next rays in the
// same lanes, and the idle lanes take new paths.  Against a launch of k_extend and one of k_shade per depth: nothing
// waits for the slowest ray of a depth, and a vertex costs no trip of its ray, hit, throughput and queue entry through
// HBM (156 bytes; the Cornell frame's shading ran at 5 TB/s).  What it costs is registers (the shading beside the
// waiting lanes' traversal state: five to six waves per SIMD instead of seven) and shading on part-filled waves.
// Bound by VALU issue (the Cornell frame: 1.0 wave64 instructions per CU per cycle).
//
// Measured, per call, before and after: the 64x36, 2-sample sphere frame 498 -> 348 us, 400x225x32 spheres 1875 ->
// 1430, Cornell 600x600x64 11490 -> 7890, RTTNW 600x600x32 6446 -> 5613, four 641x359, 1-sample mesh frames 5351 ->
// 4190, the inverse-rendering step 5054 -> 3980.

// Waves per SIMD the register budget allows.  Without sphere, media or instance code six (a few spills around the
// shading; the Cornell frame at 4, 5, 6 and 7: 9.2, 8.1, 7.8 and 7.8 ms, the 1080p mesh frame at 5, 6 and 7: 51.6,
// 49.2 and 50.0); with the sphere test five; with media or instances four (RTTNW at 4, 5 and 6: 5.6, 6.2, 7.4 ms).
constexpr int trace_waves(bool inst, bool sph, bool vol) { return inst || vol ? 4 : sph ? 5 : 6; }

// Fewest paths a wave claims, as EXTEND_CLAIM_LEAST (at 16 the 64x36, 2-sample sphere frame takes 417 us, not 344).
constexpr uint32_t TRACE_CLAIM_LEAST = 4;
// With four lanes to a path a wave holds sixteen: more at a time would leave the others idle (the four mesh preview
// frames at most 8, 16 and 32: 2.74, 2.73 and 3.18 ms; the sphere thumbnail at least 1, 2 and 4: 161, 171 and 170 us).
constexpr uint32_t QUAD_CLAIM_LEAST = 1;

// The launch's shares of the tunables, 32 lanes and 128 positions by default (worked out on the host: in the kernels they
// would hold registers).  sdf: 1 for k_trace_sdf, 2 if there is a Mandelbulb too.
inline ExtendTuning trace_tuning(ExtendTuning t, int sdf, bool quad) {
    const uint32_t n = t.refill_lanes;
    t.refill_lanes = sdf == 2 ? std::max(1u, n / 2u) : std::min(64u, sdf == 1 ? n + n / 2u : n + n / 4u);
    if (quad) t.wave_batch = std::max(QUAD_CLAIM_LEAST, t.wave_batch / 8u);
    return t;
}

// Adds the closest-hit queries that the wave's lanes counted to one of the SEGMENT_PARTS counters.  A wave's own sum fits
// 32 bits with room to spare: 2^31 paths (no GPU holds more) of a thousand vertices, over the thousands of waves that
// share them evenly, are 2^29 a wave.  (Summed in 64 bits the kernels' register allocation changed throughout: the
// Cornell frame 7.31 -> 7.61 ms, four 641x359, 1-sample mesh frames 2.70 -> 2.91.)
__device__ __forceinline__ void add_segments(SegmentCounter *segments, uint32_t lane_count) {
    for (int o = 32; o > 0; o >>= 1) lane_count += __shfl_xor(lane_count, o);
    if (__lane_id() == 0u && lane_count != 0u)
        atomicAdd(segments + SEGMENT_STRIDE * (blockIdx.x % SEGMENT_PARTS), (SegmentCounter)lane_count);
}
// first_depth 0: the paths are the chunk's slots, from their camera rays (computed here).  first_depth > 0: the paths
// are queue[0 .. *count_ptr), which k_shade kept at depth 0, from their stored rays and throughputs.
//
// QUAD: four lanes to a path (quad.hpp): all of them hold it, the first one shades and takes new paths.  Without
// instances.
template <bool QUAD, bool BATCH, bool INST, bool SPH, bool VOL, bool TEX, bool ADJOINT>
__global__ __launch_bounds__(EXT_BLOCK) __attribute__((amdgpu_waves_per_eu(trace_waves(INST, SPH, VOL)))) void k_trace(
    TraceArgs args) {
    __shared__ unsigned long long s_entry[EXT_LDS_STACK * EXT_BLOCK];
    __shared__ float s_t[3 * EXT_BLOCK];  // the paths' throughputs
    const SceneView &sv = args.sv;
    const uint32_t count = args.queue ? *args.count : args.fp.n_slots;
    // A refill shades too, so it waits for a quarter more lanes than k_extend's (at 32, 40 and 48 lanes the four mesh
    // preview frames take 4.19, 4.03 and 4.00 ms, the 1080p mesh frame 48.5, 48.3 and 49.0).  Once no path is left to
    // take, idle lanes say nothing: half of the wave's paths then wait (against refill_lanes waiting or idle, where a
    // wave with few paths shaded them one by one: the preview frames 4.24 -> 3.96 ms, the inverse-rendering step 3.97 ->
    // 3.80; at a third 4.01 and 3.77, at a twelfth 4.18 and 3.95).
    const uint32_t refill_lanes = args.tune.refill_lanes;
    const uint32_t gid = blockIdx.x * EXT_BLOCK + threadIdx.x;
    const uint32_t lane = __lane_id();
    const bool lead = !QUAD || (lane & 3u) == 0u;
    LaneStack st{(lds_u64 *)s_entry, args.overflow + gid, gridDim.x * EXT_BLOCK, 0};
    QuadStack qst{(lds_u64 *)s_entry, args.overflow + (gid & ~3u), gridDim.x * EXT_BLOCK};
    enum : int { IDLE, TRACING, HIT };  // no path; a ray in the tree; its closest hit found
    int state = IDLE;
    uint32_t slot = 0, depth = 0, n_segments = 0;
    DRay ray{};
    Best b{FLT_MAX, -1, 0u, 0u, 0u};
    LeafRange leaf;
    TravStats stats;
    WaveClaims claims(count, EXT_BLOCK / 64, QUAD ? QUAD_CLAIM_LEAST : TRACE_CLAIM_LEAST,
                      args.tune.wave_batch, args.work);
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
    dm::Key vkey{0u, 0u};
    uint32_t vpixel = 0, vsample = 0;  // VOL: kept for the free-flight draws
    for (;;) {
        unsigned long long idle = __ballot(state == IDLE);
        const unsigned long long waiting = idle | __ballot(state == HIT);
        const uint32_t n_idle = (uint32_t)__popcll(idle), n_hit = (uint32_t)__popcll(waiting) - n_idle;
        if (waiting == ~0ull || (claims.exhausted ? 2u * n_hit >= 64u - n_idle : n_idle + n_hit >= refill_lanes)) {
            const TraceArgs &A = cold_args();
            bool begin = false;
            VertexGrad grad;
            if (state == HIT && lead) {
                dm::Key key;
                uint32_t pixel, sample;
                const RequestParams *R = identify(A, &key, &pixel, &sample);
                const Col T{s_t[threadIdx.x], s_t[EXT_BLOCK + threadIdx.x], s_t[2 * EXT_BLOCK + threadIdx.x]};
                Col L{0.0f, 0.0f, 0.0f}, add{0.0f, 0.0f, 0.0f};
                if (ADJOINT) L = Col{A.pb.lr[slot], A.pb.lg[slot], A.pb.lb[slot]};
                const uint32_t at_depth = depth;
                const Best hit = b;
                begin = shade_vertex<ADJOINT, TEX, false, false>(
                    A.sv, nullptr, A.ap, grad, ray, hit.ref, &hit.t, &hit.aux, &hit.sub, false, f3{0.0f, 0.0f, 0.0f}, key,
                    pixel, sample, at_depth, BATCH ? R->ray_depth : A.fp.ray_depth, BATCH ? R->skybox : A.sv.skybox,
                    BATCH ? R->sky_image : A.sv.sky_image, T, L, add, [&](const DRay &nr, const Col &t) {
                        ray = ray_from_dir(nr.o, nr.d);
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
            idle = __ballot(state == IDLE && !begin && lead);
            if (!claims.exhausted && idle != 0ull) {
                const uint32_t q = claims.hand_out(idle);
                if (state == IDLE && !begin && lead && q != 0xffffffffu) {
                    slot = A.queue ? (uint32_t)A.queue[q] : q;
                    depth = A.first_depth;
                    Col T{1.0f, 1.0f, 1.0f};
                    if (A.first_depth == 0u) {
                        dm::Key key;
                        uint32_t pixel, sample;
                        const RequestParams *R = identify(A, &key, &pixel, &sample);
                        const DRay c = BATCH ? camera_ray(R->vp, R->width, R->height, R->sdim, key, pixel, sample)
                                             : camera_ray(A.fp.vp, A.fp.width, A.fp.height, A.fp.sdim, key, pixel, sample);
                        ray = ray_from_dir(c.o, c.d);
                    } else {
                        ray = ray_from_dir(f3{A.pb.ox[slot], A.pb.oy[slot], A.pb.oz[slot]},
                                           f3{A.pb.dx[slot], A.pb.dy[slot], A.pb.dz[slot]});
                        T = Col{A.pb.tr[slot], A.pb.tg[slot], A.pb.tb[slot]};
                    }
                    s_t[threadIdx.x] = T.r;
                    s_t[EXT_BLOCK + threadIdx.x] = T.g;
                    s_t[2 * EXT_BLOCK + threadIdx.x] = T.b;
                    begin = true;
                }
            }
            if (QUAD) {  // the first lane's path to all four
                state = (int)quad_perm<QUAD_FIRST>((uint32_t)state);
                begin = quad_perm<QUAD_FIRST>(begin ? 1u : 0u) != 0u;
                if (begin) {
                    slot = quad_perm<QUAD_FIRST>(slot);
                    depth = quad_perm<QUAD_FIRST>(depth);
                    ray.o = f3{quad_perm<QUAD_FIRST>(ray.o.x), quad_perm<QUAD_FIRST>(ray.o.y),
                               quad_perm<QUAD_FIRST>(ray.o.z)};
                    ray.d = f3{quad_perm<QUAD_FIRST>(ray.d.x), quad_perm<QUAD_FIRST>(ray.d.y),
                               quad_perm<QUAD_FIRST>(ray.d.z)};
                    ray.inv = f3{quad_perm<QUAD_FIRST>(ray.inv.x), quad_perm<QUAD_FIRST>(ray.inv.y),
                                 quad_perm<QUAD_FIRST>(ray.inv.z)};
                }
            }
            if (begin) {
                int32_t root = A.sv.root;
                if (BATCH) root = A.bv.reqs[A.bv.slot_req[slot]].root;
                if (VOL) (void)identify(A, &vkey, &vpixel, &vsample);
                if (INST) {  // finish_instance reloads the world ray
                    A.pb.ox[slot] = ray.o.x;
                    A.pb.oy[slot] = ray.o.y;
                    A.pb.oz[slot] = ray.o.z;
                    A.pb.dx[slot] = ray.d.x;
                    A.pb.dy[slot] = ray.d.y;
                    A.pb.dz[slot] = ray.d.z;
                }
                b = Best{FLT_MAX, -1, 0u, 0u, 0u};
                if (QUAD) {
                    qst.sp = 0;
                    qst.has = root >= 0;
                    qst.code = root;
                    qst.t = 0.0f;
                } else {
                    st.sp = 0;
                    st.top_valid = false;
                    if (root >= 0) st.push(root, -__builtin_inff());
                    leaf.code = 0;
                }
                state = TRACING;
                if (lead) ++n_segments;
            }
        }
        if (!__any(state == TRACING)) {
            if (claims.exhausted && !__any(state == HIT)) break;
            continue;
        }
        if (state == TRACING) {
            if (QUAD) {
                traverse_quad_pass<SPH, VOL>(sv, ray, b, qst, vkey, vpixel, vsample, depth);
                if (!qst.has && qst.sp == 0) state = HIT;
            } else {
                traverse_pass<INST, SPH, VOL>(sv, args.pb, slot, ray, b, leaf, st, vkey, vpixel, vsample, depth, stats);
                if (st.sp == 0 && leaf.code == 0) state = HIT;
            }
        }
    }
    stats.flush();
    add_segments(args.segments, n_segments);
}
