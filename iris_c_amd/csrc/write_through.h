/* Stores of results that leave the L2 as they are issued (sc0 sc1). A kernel that stores plainly leaves its results dirty in the L2s,
 * which write them back at its end, in front of the next launch. Each kernel that uses these says what it measured. */
#ifndef IRIS_WRITE_THROUGH_H
#define IRIS_WRITE_THROUGH_H

/* 16 or 8 bytes. The compiler does not know that the statement is a store: the wait states stand for those it would place before
 * the registers are written again. */
template <typename V> __device__ __forceinline__ void store_through(void *p, V v) {
    if constexpr (sizeof(V) == 16) asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
    else asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

#endif
