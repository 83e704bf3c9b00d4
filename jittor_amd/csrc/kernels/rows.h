// Fused groups and the reductions between them in one pass over the rows of a [rows, cols] iteration space: a normalisation or a
// softmax, forward and backward (the reference's executor lets element, broadcast and reduce ops share a group,
// python/jittor/src/executor.cc:555; member kernels ops/reduce_op.cc:374-399 and those of fused.h).
//
// G lanes hold one row in registers, NV packs of VEC adjacent elements each: pack t of lane l covers the columns (t * G + l) * VEC.
// Every full-size input is read once and every full-size result written once, whatever the number of reductions between them: HBM
// bounds it (us, part by part / so, floor at the rate of a copy: layer normalisation forward and backward 16384 x 1024 float32 287 / 50,
// 43; 65536 x 64 86 / 17.5, 11; 64 x 16384 51 / 22; softmax forward and backward 16384 x 512 109 / 21.4, 21; 8000 x 1001 114 / 21.5, 20;
// 1000 x 777 40 / 5.4).  A row of more than 8 elements a lane keeps the values per column out of its registers and loads them where
// they are used (16 elements of 16 bits a lane, 1024 lanes, two scales and their sums: 86 / 22).
// The host generates from the group's ops:
//   MJT_ROWS_SCALARS    by-value scalars and single elements
//   MJT_ROWS_COLS       packs of the inputs that have one value per column, loaded once for all rows of the workgroup
//   MJT_ROWS_LOADS      the row's packs of the full-size inputs, its values of the inputs that have one per row
//   MJT_ROWS_BODY       reductions in the order of their dependence: accumulate over the lane's elements, combine over the row's lanes;
//                       the ops of one value per row; the element ops behind the last reduction, stores, column sums
//   MJT_ROWS_SUMS       accumulators of the column sums;  NSUMS their number, MJT_ROWS_SUM(j) the j-th
//   LEVELS, MOST        rounds of reductions a row, most reductions in one
//   TAIL                1: cols is less than G * NV * VEC
// Up to 64 lanes combine by shuffles; more (whole waves) through LDS, where a slot is written again only two rows later, behind
// another barrier.  A column sum stays in the lane that owns the column while the workgroup walks over its rows; the row groups of the
// workgroup are added up in LDS, the workgroups' results by the fold kernel below.

struct Params { void* a[NPARAM]; };   // 8-byte words; typed as pointers so loads/stores use the global address space
// a[0] rows  a[1] cols  a[2] rcount of mean (double bits)  a[3] partial column sums [workgroup][sum][cols]

#define RPB (BLOCK / G)                  // rows a workgroup works on at once
#define GW (G > 64 ? G / 64 : 1)         // waves that share a row

#ifndef FOLD
template <class T> __device__ __forceinline__ T mjt_rows_xor(T v, int off) {
    int t = 0;
    __builtin_memcpy(&t, &v, sizeof(T));
    t = __shfl_xor(t, off, 64);
    __builtin_memcpy(&v, &t, sizeof(T));
    return v;
}

extern "C" __global__ __launch_bounds__(BLOCK) void ENTRY(Params p) {
    const int rows = (int)(long long)p.a[0], cols = (int)(long long)p.a[1];
    const float rcount = (float)__longlong_as_double((long long)(unsigned long long)p.a[2]);
    const int tid = threadIdx.x, lane = tid % G, sub = tid / G;
    const bool inside = ((NV - 1) * G + lane) * VEC < cols;             // of the lane's last pack
    const int last = inside ? ((NV - 1) * G + lane) * VEC : cols - VEC;
    (void)rcount, (void)inside, (void)last;
#if GW > 1
    __shared__ float slots[2][LEVELS][MOST][BLOCK / 64];
#endif
    MJT_ROWS_SCALARS
    MJT_ROWS_COLS
    MJT_ROWS_SUMS
    int turn = 0;
#pragma unroll 1
    for (int row0 = (int)blockIdx.x * RPB; row0 < rows; row0 += (int)gridDim.x * RPB, turn ^= 1) {
        const bool mine = row0 + sub < rows;                 // (a row group past the end works on the last row and keeps nothing)
        const int row = mine ? row0 + sub : rows - 1;
        const long long base = (long long)row * cols;
        MJT_ROWS_LOADS
        MJT_ROWS_BODY
    }
#if NSUMS
    float* __restrict__ part = (float*)p.a[3] + (long long)blockIdx.x * NSUMS * cols;
#if RPB > 1
    __shared__ float meet[RPB][G * NV * VEC];
#endif
#pragma unroll
    for (int j = 0; j < NSUMS; j++) {
#if RPB > 1
        if (j) __syncthreads();
#pragma unroll
        for (int t = 0; t < NV; t++)
#pragma unroll
            for (int k = 0; k < VEC; k++) meet[sub][(t * G + lane) * VEC + k] = sums[j][t][k];
        __syncthreads();
        for (int c = tid; c < cols; c += BLOCK) {
            float s[RPB];
#pragma unroll
            for (int q = 0; q < RPB; q++) s[q] = meet[q][c];
#pragma unroll
            for (int off = RPB / 2; off > 0; off /= 2)
#pragma unroll
                for (int q = 0; q < off; q++) s[q] += s[q + off];
            part[(long long)j * cols + c] = s[0];
        }
#else
#pragma unroll
        for (int t = 0; t < NV; t++)
#pragma unroll
            for (int k = 0; k < VEC; k++)
                if (!TAIL || (t * G + lane) * VEC < cols) part[(long long)j * cols + (t * G + lane) * VEC + k] = sums[j][t][k];
#endif
    }
#endif
}
#else
// The workgroups' partial sums added up: 32 columns and 32 groups of workgroups per workgroup, a column's groups meet in LDS.
// a[0] workgroups  a[1] cols  a[2] partial sums  a[3 ..] results, their types TOUT(j)
extern "C" __global__ __launch_bounds__(1024) void ENTRY(Params p) {
    const int n = (int)(long long)p.a[0], cols = (int)(long long)p.a[1];
    const int c = (int)blockIdx.x * 32 + (threadIdx.x & 31), g = threadIdx.x >> 5, j = blockIdx.y;
    const float* __restrict__ part = (const float*)p.a[2] + (long long)j * cols + c;
    __shared__ float meet[32][33];
    float s[8] = {};                         // eight loads on their way, eight short chains of roundings
    if (c < cols) {
        int b = g;
        for (; b + 7 * 32 < n; b += 8 * 32)
#pragma unroll
            for (int q = 0; q < 8; q++) s[q] += part[(long long)(b + q * 32) * NSUMS * cols];
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (b + q * 32 < n) s[q] += part[(long long)(b + q * 32) * NSUMS * cols];
    }
    meet[g][threadIdx.x & 31] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
#pragma unroll
    for (int off = 16; off > 0; off /= 2) {
        if (g < off) meet[g][threadIdx.x & 31] += meet[g + off][threadIdx.x & 31];
        __syncthreads();
    }
    if (g == 0 && c < cols) {
        const float all = meet[0][threadIdx.x];
        MJT_FOLD_STORE
    }
}
#endif
