// Byte places of what the dequantising tiles (gemm_dq_slots.h) load, apart from them so that the host can check them: row r of a
// tile, step s of K (64 of it), lanes 0 .. 31 (fq 0) and 32 .. 63 (fq 1). The tiles ask for steps past the slice's last one (kl),
// whose values they never multiply: those take the last step's place, so no load lies past its operand. (A buffer descriptor's
// range check does not stand in for that: the step is in the scalar offset, which the check need not include.)
#pragma once

namespace omx {

constexpr unsigned ds_step(int s, int kl) { return (unsigned)(s < kl ? s : kl); }
// activations, fp16 [rows][Kp]: piece xc (16 bytes) of the step
constexpr unsigned ds_x_at(unsigned r, unsigned Kp, unsigned xc) { return 2u * (r * Kp + 8u * xc); }
constexpr unsigned ds_x_step(int s, int kl) { return 128u * ds_step(s, kl); }
// codes or high bits of `block` bytes a super-block, the row's first super-block sb0: piece 2 s + fq
constexpr unsigned ds_w_at(unsigned sb0, unsigned block, unsigned fq) { return sb0 * block + block / 8u * fq; }
constexpr unsigned ds_w_step(int s, int kl, unsigned block) { return block / 4u * ds_step(s, kl); }
// fp16 scale of piece lt (which counts on past a super-block's eight) of super-block sb, 16 bytes of scales each
constexpr unsigned ds_scale_at(unsigned sb, unsigned lt) { return 16u * sb + 2u * (lt < 7u ? lt : 7u); }

}  // namespace omx
