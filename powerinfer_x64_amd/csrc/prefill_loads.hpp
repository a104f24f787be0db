// prefill_loads.hpp -- the direct global -> LDS loads of prefill_fa_kernel (prefill.hip): how many
// each wavefront issues per unit (K of one key tile, V of the one before), and the vmcnt its waits
// may leave in flight.  Apart so that a host walk can check the waits (tests/cpp).
#pragma once

namespace pi {

// wavefronts and LDS unit buffers of a workgroup
template <int D> struct PrefillCfg;
template <> struct PrefillCfg<64> { static constexpr int NW = 8, NB = 4; };
template <> struct PrefillCfg<128> { static constexpr int NW = 8, NB = 4; };
template <> struct PrefillCfg<256> { static constexpr int NW = 4, NB = 2; };

template <int D, bool PG>
struct PrefillLoads {
    static constexpr int BN = 64;                // keys per tile
    static constexpr int NW = PrefillCfg<D>::NW;
    static constexpr int KS = D + 8;             // K [key][dim] row stride (elements): 16 bytes of padding
    static constexpr int KCH = KS / 8;           // 16-byte chunks per K row
    // loads of 1 KB per K tile: the padded rows (9, 17 or 33); paged, D / 8 (one per 16-byte chunk)
    static constexpr int K_INSTR = PG ? D / 8 : BN * KCH / 64;
    static constexpr int KJ = (K_INSTR + NW - 1) / NW;  // K loads per wavefront, at most
    static constexpr int V_INSTR = BN * D * 2 / 1024;   // loads of 1 KB per V tile (8, 16 or 32)
    static constexpr int VJ = V_INSTR / NW;             // V loads per wavefront
    // paged, 8 wavefronts: waves 0-3 issue the shares of two waves, the others none
    static constexpr int LPD = (PG && NW == 8) ? 2 : 1;
    // K load i of a tile is wave i % NW's, so only the first K_INSTR % NW waves have KJ of them
    static constexpr int K_MOST = K_INSTR % NW;
    // A wave's loads of a unit that has both tiles: the count that a wait for the unit before it
    // leaves in flight.  A count above the loads really issued would wait for nothing.
    static constexpr int unit_loads(int wave) {
        return LPD * (K_INSTR / NW + (!PG && wave < K_MOST ? 1 : 0) + VJ);
    }
    static_assert(V_INSTR % NW == 0 && (PG ? K_MOST == 0 : K_MOST == 1), "unit_loads");
};

}  // namespace pi
