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

// first_depth 0: the paths are the chunk's slots, from their camera rays (computed here).  first_depth > 0: the paths
// are queue[0 .. *count_ptr), which k_shade kept at depth 0, from their stored rays and throughputs.
template <bool BATCH, bool INST, bool SPH, bool VOL, bool TEX, bool ADJOINT>
__global__ __launch_bounds__(EXT_BLOCK) __attribute__((amdgpu_waves_per_eu(trace_waves(INST, SPH, VOL)))) void k_trace(
    SceneView sv, FrameParams fp, PathBuffers pb, const int32_t *queue, const uint32_t *count_ptr,
    uint32_t first_depth, int2 *overflow, uint32_t *work, uint32_t *segments, ExtendTuning tune, AdjointParams ap,
    BatchView bv) {
    __shared__ unsigned long long s_entry[EXT_LDS_STACK * EXT_BLOCK];
    __shared__ float s_t[3 * EXT_BLOCK];  // the paths' throughputs
    const uint32_t count = queue ? *count_ptr : fp.n_slots;
    // A refill shades too, so it waits for a quarter more lanes than k_extend's (at 32, 40 and 48 lanes the four mesh
    // preview frames take 4.19, 4.03 and 4.00 ms, the 1080p mesh frame 48.5, 48.3 and 49.0).
    const uint32_t refill_lanes = tune.refill_lanes + tune.refill_lanes / 4u < 64u
                                      ? tune.refill_lanes + tune.refill_lanes / 4u
                                      : 64u;
    const uint32_t gid = blockIdx.x * EXT_BLOCK + threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t copy = ADJOINT ? blockIdx.x % ap.copies : 0u;
    LaneStack st{(lds_u64 *)s_entry, overflow + gid, gridDim.x * EXT_BLOCK, 0};
    enum : int { IDLE, TRACING, HIT };  // no path; a ray in the tree; its closest hit found
    int state = IDLE;
    uint32_t slot = 0, depth = 0, n_segments = 0;
    DRay ray{};
    Best b{FLT_MAX, -1, 0u, 0u, 0u};
    int32_t leaf = 0;
    int leaf_i = 0, leaf_n = 0;
    float leaf_t = 0.0f;
    uint32_t batch_next = 0, batch_end = 0;
    bool exhausted = false;
    WaveClaims claims(count, EXT_BLOCK / 64, TRACE_CLAIM_LEAST, tune.wave_batch, work);
    // the path's RNG key, pixel and sample, and in a batch its request
    auto identify = [&](dm::Key *key, uint32_t *pixel, uint32_t *sample) -> const RequestParams * {
        if (BATCH) {
            const RequestParams *R = bv.reqs + bv.slot_req[slot];
            const uint32_t l = slot - R->slot_base;
            *key = dm::Key{R->key0, R->key1};
            *pixel = l / R->n_spp;
            *sample = R->s0 + l % R->n_spp;
            return R;
        }
        *key = dm::Key{fp.key0, fp.key1};
        *pixel = slot / fp.n_spp;
        *sample = fp.s0 + slot % fp.n_spp;
        return nullptr;
    };
    dm::Key vkey{fp.key0, fp.key1};
    uint32_t vpixel = 0, vsample = 0;  // VOL: kept for the free-flight draws
    for (;;) {
        unsigned long long idle = __ballot(state == IDLE);
        const unsigned long long waiting = idle | __ballot(state == HIT);
        if (waiting == ~0ull || (uint32_t)__popcll(waiting) >= refill_lanes) {
            bool begin = false;
            if (state == HIT) {
                dm::Key key;
                uint32_t pixel, sample;
                const RequestParams *R = identify(&key, &pixel, &sample);
                const Col T{s_t[threadIdx.x], s_t[EXT_BLOCK + threadIdx.x], s_t[2 * EXT_BLOCK + threadIdx.x]};
                Col L{0.0f, 0.0f, 0.0f}, add{0.0f, 0.0f, 0.0f};
                if (ADJOINT) L = Col{pb.lr[slot], pb.lg[slot], pb.lb[slot]};
                const uint32_t at_depth = depth;
                const Best hit = b;
                begin = shade_vertex<ADJOINT, TEX, false, false>(
                    sv, nullptr, ap, copy, ray, hit.ref, &hit.t, &hit.aux, &hit.sub, false, f3{0.0f, 0.0f, 0.0f}, key,
                    pixel, sample, at_depth, BATCH ? R->ray_depth : fp.ray_depth, BATCH ? R->skybox : sv.skybox,
                    BATCH ? R->sky_image : sv.sky_image, T, L, add, [&](const DRay &nr, const Col &t) {
                        ray = ray_from_dir(nr.o, nr.d);
                        s_t[threadIdx.x] = t.r;
                        s_t[EXT_BLOCK + threadIdx.x] = t.g;
                        s_t[2 * EXT_BLOCK + threadIdx.x] = t.b;
                        ++depth;
                    });
                const bool adds = !(add.r == 0.0f && add.g == 0.0f && add.b == 0.0f);
                if (!ADJOINT && at_depth != 0u && adds) L = Col{pb.lr[slot], pb.lg[slot], pb.lb[slot]};
                if (!ADJOINT) L = L + add;
                if (ADJOINT || at_depth == 0u || adds) {
                    pb.lr[slot] = L.r;
                    pb.lg[slot] = L.g;
                    pb.lb[slot] = L.b;
                }
                state = IDLE;
            }
            idle = __ballot(state == IDLE && !begin);
            if (!exhausted && idle != 0ull) {
                const uint32_t n = (uint32_t)__popcll(idle);
                const uint32_t r = batch_end - batch_next;
                uint32_t nb = 0, nb_end = 0;
                if (r < n && !claims.last) claims.take(__ffsll((long long)idle) - 1, &nb, &nb_end);
                const uint32_t idx = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                uint32_t q = 0xffffffffu;
                if (idx < r) q = batch_next + idx;
                else if (idx - r < nb_end - nb) q = nb + (idx - r);
                if (r >= n) {
                    batch_next += n;
                } else {
                    const uint32_t from_new = (n - r < nb_end - nb) ? n - r : nb_end - nb;
                    batch_next = nb + from_new;
                    batch_end = nb_end;
                }
                if (claims.last && batch_next == batch_end) exhausted = true;
                if (state == IDLE && !begin && q != 0xffffffffu) {
                    slot = queue ? (uint32_t)queue[q] : q;
                    depth = first_depth;
                    Col T{1.0f, 1.0f, 1.0f};
                    if (first_depth == 0u) {
                        dm::Key key;
                        uint32_t pixel, sample;
                        const RequestParams *R = identify(&key, &pixel, &sample);
                        const DRay c = BATCH ? camera_ray(R->vp, R->width, R->height, R->sdim, key, pixel, sample)
                                             : camera_ray(fp.vp, fp.width, fp.height, fp.sdim, key, pixel, sample);
                        ray = ray_from_dir(c.o, c.d);
                    } else {
                        ray = ray_from_dir(f3{pb.ox[slot], pb.oy[slot], pb.oz[slot]},
                                           f3{pb.dx[slot], pb.dy[slot], pb.dz[slot]});
                        T = Col{pb.tr[slot], pb.tg[slot], pb.tb[slot]};
                    }
                    s_t[threadIdx.x] = T.r;
                    s_t[EXT_BLOCK + threadIdx.x] = T.g;
                    s_t[2 * EXT_BLOCK + threadIdx.x] = T.b;
                    begin = true;
                }
            }
            if (begin) {
                int32_t root = sv.root;
                if (BATCH) root = bv.reqs[bv.slot_req[slot]].root;
                if (VOL) (void)identify(&vkey, &vpixel, &vsample);
                if (INST) {  // finish_instance reloads the world ray
                    pb.ox[slot] = ray.o.x;
                    pb.oy[slot] = ray.o.y;
                    pb.oz[slot] = ray.o.z;
                    pb.dx[slot] = ray.d.x;
                    pb.dy[slot] = ray.d.y;
                    pb.dz[slot] = ray.d.z;
                }
                b = Best{FLT_MAX, -1, 0u, 0u, 0u};
                st.sp = 0;
                st.top_valid = false;
                if (root >= 0) st.push(root, -__builtin_inff());
                leaf = 0;
                state = TRACING;
                ++n_segments;
            }
        }
        if (!__any(state == TRACING)) {
            if (exhausted && !__any(state == HIT)) break;
            continue;
        }
        if (state == TRACING) {  // k_extend's loops
            bool stalled = leaf != 0 && ((uint32_t)leaf & LEAF_CODE_ITEMS) && leaf_i > 0;
            for (;;) {
                const unsigned long long searching = __ballot(leaf == 0 && st.sp > 0);
                if (searching == 0ull) break;
                if ((uint32_t)__popcll(searching) <= EXTEND_INNER_EXIT && __any(leaf != 0)) break;
                if (stalled || st.sp == 0) continue;
                int32_t code;
                float tent;
                st.pop(&code, &tent);
                if (!(tent <= b.t * BOX_SLACK)) {
                    if (INST && tent != tent) {
                        if (leaf != 0) {
                            st.push(code, tent);
                            stalled = true;
                        } else {
                            finish_instance(sv, pb, slot, code, ray, b, st);
                        }
                    }
                    continue;
                }
                if (code < 0) {
                    if (leaf != 0) {
                        st.push(code, tent);
                        stalled = true;
                        continue;
                    }
                    leaf = code;
                    leaf_i = 0;
                    leaf_n = (int)(((uint32_t)code >> 27) & 7u) + 1;
                    leaf_t = tent;
                    continue;
                }
                expand(sv, ray, b.t, code, st);
            }
            do {
                if (leaf != 0) {
                    if (leaf_test<INST, SPH, VOL>(sv, ray, leaf, leaf_i, leaf_t, b, st, vkey, vpixel, vsample, depth) ||
                        ++leaf_i == leaf_n)
                        leaf = 0;
                }
            } while ((uint32_t)__popcll(__ballot(leaf != 0)) > EXTEND_PRIM_EXIT);
            if (st.sp == 0 && leaf == 0) state = HIT;
        }
    }
    // the wave's closest-hit queries, added to one of SEGMENT_PARTS counters a line apart
    for (int o = 32; o > 0; o >>= 1) n_segments += __shfl_xor(n_segments, o);
    if (lane == 0u && n_segments != 0u) atomicAdd(segments + 32 * (blockIdx.x % SEGMENT_PARTS), n_segments);
}
