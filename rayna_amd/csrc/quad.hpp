// Closest-hit traversal with four lanes to a ray (included by kernels.hip inside its anonymous namespace, after
// traverse.hpp), for launches too small to give every lane a ray of its own.
//
// There the time is one ray's serial chain of instructions: with a lane to a ray a node expansion is some 175 vector
// instructions and a leaf's primitives are tested one after another.  Here the four lanes of a quad hold the same ray
// and closest hit; each tests one child box of a node, or one primitive of a leaf range, and quad permutations of the
// lanes order the children and merge the hits.  An expansion is some 60 instructions, a range of four primitives one
// test.  The quad's stack is depth-first (packet_need bounds it).  Results are traverse_pass's: culling is
// conservative and the closest hit, ties to the higher rank, does not depend on the order of the tests.

// Bound by the longest path's chain of instructions and node fetches.  Per call, a lane and four lanes to a ray: the
// 64x36, 2-sample sphere frame 287 -> 161 us, four 641x359, 1-sample mesh frames 3.60 -> 2.70 ms; full launches are
// slower (the 1080p mesh frame 44.7 -> 54.1 ms, Cornell 7.4 -> 18.3: the children's order is worked out four times).

constexpr int QUAD_LDS_STACK = 4 * EXT_LDS_STACK;  // entries per quad in LDS, in the space of its lanes' columns

constexpr int QUAD_XOR1 = 0xB1, QUAD_XOR2 = 0x4E, QUAD_ROT1 = 0x39, QUAD_ROT3 = 0x93, QUAD_FIRST = 0x00;
// The value of another lane of the quad (lanes of a quad are active together).
template <int PERM>
__device__ __forceinline__ uint32_t quad_perm(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, PERM, 0xf, 0xf, true);
}
template <int PERM>
__device__ __forceinline__ float quad_perm(float v) {
    return __uint_as_float(quad_perm<PERM>(__float_as_uint(v)));
}
__device__ __forceinline__ uint32_t quad_or(uint32_t v) {
    v |= quad_perm<QUAD_XOR1>(v);
    return v | quad_perm<QUAD_XOR2>(v);
}
// The quad's four bits of a ballot.
__device__ __forceinline__ uint32_t quad_bits(unsigned long long mask) {
    return (uint32_t)(mask >> (__lane_id() & 60u)) & 15u;
}

// Between one lane's store of a stack entry and another lane's load of it, and between loads and a store that takes
// their place: keeps the compiler from moving either across (the wave's own accesses to LDS and memory stay in order,
// so this costs no instruction).
__device__ __forceinline__ void quad_stack_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A quad's traversal: the entry it holds (code, entry distance) and the stack below it.
struct QuadStack {
    lds_u64 *s_entry;
    int2 *g;  // the overflow column of the quad's first lane
    uint32_t stride;
    int sp = 0;
    bool has = false;
    int32_t code = 0;
    float t = 0.0f;
    __device__ __forceinline__ void store(int i, int32_t n, float v) {
        if (i < QUAD_LDS_STACK) s_entry[i * (EXT_BLOCK / 4) + threadIdx.x / 4] = stack_word(n, v);
        else g[(size_t)(i - QUAD_LDS_STACK) * stride] = make_int2(n, __float_as_int(v));
    }
    __device__ __forceinline__ void pop() {
        --sp;
        if (sp < QUAD_LDS_STACK) {
            const unsigned long long e = s_entry[sp * (EXT_BLOCK / 4) + threadIdx.x / 4];
            code = (int32_t)(uint32_t)e;
            t = __uint_as_float((uint32_t)(e >> 32));
        } else {
            const int2 e = g[(size_t)(sp - QUAD_LDS_STACK) * stride];
            code = e.x;
            t = __int_as_float(e.y);
        }
    }
};

// Expands the inner node the quad holds: the nearest child its ray hits becomes the entry it holds, the others go on
// its stack, far to near.  Distances are ordered as bit patterns with the lane in their two lowest bits (they are at
// least T_MIN, and lowering one by three units culls no more).
__device__ __forceinline__ void expand_quad(const SceneView &sv, const DRay &ray, float best, QuadStack &st) {
    const uint32_t c = __lane_id() & 3u;
    const float *np = reinterpret_cast<const float *>(sv.nodes + st.code) + c;
    const float lx = np[0], ly = np[4], lz = np[8], hx = np[12], hy = np[16], hz = np[20];
    const int32_t code = reinterpret_cast<const int32_t *>(np)[28];  // the slot's entry code (device node copy)
    const float tx1 = (lx - ray.o.x) * ray.inv.x, tx2 = (hx - ray.o.x) * ray.inv.x;
    float t0 = fminf(tx1, tx2), t1 = fmaxf(tx1, tx2);
    const float ty1 = (ly - ray.o.y) * ray.inv.y, ty2 = (hy - ray.o.y) * ray.inv.y;
    t0 = fmaxf(t0, fminf(ty1, ty2));
    t1 = fminf(t1, fmaxf(ty1, ty2));
    const float tz1 = (lz - ray.o.z) * ray.inv.z, tz2 = (hz - ray.o.z) * ray.inv.z;
    t0 = fmaxf(t0, fminf(tz1, tz2));
    t1 = fminf(t1, fmaxf(tz1, tz2));
    const float lo = fmaxf(t0, T_MIN), hi = fminf(t1, best);
    const bool hit = code != ENTRY_NONE && lo <= hi * BOX_SLACK;
    const uint32_t key = hit ? (__float_as_uint(lo) & ~3u) | c : 0u;
    const int n = __popc(quad_bits(__ballot(hit)));
    const int below = (quad_perm<QUAD_ROT1>(key) > key ? 1 : 0) + (quad_perm<QUAD_XOR2>(key) > key ? 1 : 0) +
                      (quad_perm<QUAD_ROT3>(key) > key ? 1 : 0);  // children farther than this lane's
    const bool nearest = hit && below == n - 1;
    const float t = __uint_as_float(key & ~3u);
    quad_stack_order();
    if (hit && !nearest) st.store(st.sp + below, code, t);
    quad_stack_order();
    st.has = n > 0;
    st.sp += n > 0 ? n - 1 : 0;
    st.code = (int32_t)quad_or(nearest ? (uint32_t)code : 0u);
    st.t = __uint_as_float(quad_or(nearest ? key & ~3u : 0u));
}

// One pass over the wave's active quads: inner nodes, until few lanes still search for a leaf range while some quad
// holds one, then the held ranges.  A quad's traversal has ended when it holds no entry and its stack is empty.
template <bool SPH, bool VOL>
__device__ __forceinline__ void traverse_quad_pass(const SceneView &sv, DRay &ray, Best &b, QuadStack &st,
                                                   const dm::Key &key, uint32_t pixel, uint32_t sample,
                                                   uint32_t bounce) {
    for (;;) {
        const bool searching = st.has ? st.code >= 0 : st.sp > 0;
        const unsigned long long m = __ballot(searching);
        if (m == 0ull) break;
        if ((uint32_t)__popcll(m) <= EXTEND_INNER_EXIT && __any(st.has && st.code < 0)) break;
        if (!searching) continue;
        if (!st.has) {
            st.pop();
            if (!(st.t <= b.t * BOX_SLACK)) continue;  // culled
            st.has = true;
            if (st.code < 0) continue;
        }
        expand_quad(sv, ray, b.t, st);
    }
    if (st.has && st.code < 0) {
        const uint32_t c = __lane_id() & 3u;
        const int n = (int)(((uint32_t)st.code >> 27) & 7u) + 1;
        const int32_t start = (int32_t)((uint32_t)st.code & LEAF_CODE_START);
        const bool items = ((uint32_t)st.code & LEAF_CODE_ITEMS) != 0u;
        LaneStack unused{nullptr, nullptr, 0, 0};  // leaf_test<false, ...> pushes only for links, handled here
        Best mine = b;
        for (int i = (int)c; i - (int)c < n; i += 4) {
            bool link = false;
            if (i < n) {
                link = items && sv.items[start + i].kind == ITEM_LINK;
                if (!link)
                    (void)leaf_test<false, SPH, VOL>(sv, ray, st.code, i, st.t, mine, unused, key, pixel, sample, bounce);
            }
            if (items) {
                const uint32_t links = quad_bits(__ballot(link));
                quad_stack_order();
                if (link) st.store(st.sp + __popc(links & ((1u << c) - 1u)), sv.items[start + i].index, st.t);
                quad_stack_order();
                st.sp += __popc(links);
            }
        }
        if (__any(mine.t < b.t || mine.rank != b.rank)) {  // the best of the quad's four
            auto merge = [&](float t, int32_t rank, uint32_t ref, uint32_t aux) {
                if (t < mine.t || (t == mine.t && rank > mine.rank)) mine = Best{t, rank, ref, aux, 0u};
            };
            merge(quad_perm<QUAD_XOR1>(mine.t), (int32_t)quad_perm<QUAD_XOR1>((uint32_t)mine.rank),
                  quad_perm<QUAD_XOR1>(mine.ref), quad_perm<QUAD_XOR1>(mine.aux));
            merge(quad_perm<QUAD_XOR2>(mine.t), (int32_t)quad_perm<QUAD_XOR2>((uint32_t)mine.rank),
                  quad_perm<QUAD_XOR2>(mine.ref), quad_perm<QUAD_XOR2>(mine.aux));
            b = mine;
        }
        st.has = false;
    }
}
