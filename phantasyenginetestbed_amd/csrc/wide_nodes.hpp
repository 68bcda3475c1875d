// Four-wide nodes of an SBVH: the device-side form of the tree that the traversal kernels walk.
//
// A wide node merges a binary node with up to two of its descendants, so one 112-B record decides
// four boxes where castRay's binary nodes take three dependent loads. Hits stay castRay's bit for
// bit because
//   - castRay's order does not depend on the ray: at a node, the leaf children are tested (left,
//     then right), then the right inner child's subtree, then the left one's. The slots of a wide
//     node are kept in that order, so taking the slots in order is castRay's order;
//   - every child box lies inside its parent's (but see kWideLoose), and for a ray with an origin within 2^126
//     a child that passes the box predicate at some closest t implies that its ancestors passed theirs at
//     the larger t of that earlier moment: the binary node decisions that a wide node leaves out can never
//     have been negative. Without NaN slab values, because rounding is monotonic. With them (0 * inf: a
//     direction component of zero, the origin on a plane of the box) castRay's min and max, which return
//     their first operand, reject the box where the axis is x, or the plane the maximum and the box not
//     flat there, and ignore the axis otherwise. Inside a box that is rejected so, only a box that is flat
//     at that maximum, in y or z, is not rejected too; a binary node with such a child is not left out.
//     (A NaN component makes every box's values of its axis NaN.)
//   - a leaf is decided with the closest t it would be decided with by castRay: its entry distance
//     is kept with the pending slot and compared when the slot is taken. Two leaves of one parent
//     are decided together, before either is tested (kWidePair).
// Trees where this does not hold (bounds outside +-2^126 or NaN, inverted child boxes, more than
// kWideMaxPending slots pending at once) get no wide nodes and are traversed binary, as rays with
// origins beyond 2^126 are.
#pragma once

#include <cstdint>
#include <vector>

#include "../../include/phx.h"

namespace phx {

// One slot's reference: an inner slot holds the wide node's index; a leaf slot holds kWideLeaf,
// its first triangle and (bits 28-29) its triangle count if that is 1 to 3, else 0 -- the
// end marker of the triangle array ends it then. kWidePair: the next slot is the sibling leaf.
constexpr uint32_t kWideLeaf = 0x80000000u;
constexpr uint32_t kWidePair = 0x40000000u;
// An inner slot whose node's child boxes stick out of its own (of a tree made elsewhere, by a rounding):
// neither that node nor its parent is merged into another, so that it is decided when castRay decides it,
// and it is taken whatever its entry distance and the closest t are by then, as castRay takes it; its
// children are decided by themselves. Trees with such slots are loose ones.
constexpr uint32_t kWideLoose = kWidePair;
constexpr uint32_t kWideIndex = 0x0FFFFFFFu;
constexpr uint32_t kWideCountShift = 28u;

// Pending slots a traversal may hold (the kernels' stacks hold this many 8-byte entries).
constexpr uint32_t kWideMaxPending = 60u;

// 128 B, one cache line: a 32-B record per slot, so that four lanes read one slot each. Slots 0 to 2
// repeat slot 3's max.xyz in their last words, so that one lane reads the whole node in its first seven
// 16-B words. Empty slots have NaN boxes, which no ray passes.
struct WideNode {
	struct Slot {
		float min[3];
		uint32_t ref;
		float max[3];
		float lastMax;  // slot i < 3: slot[3].max[i]
	} slot[4];
	WideNode() {}  // left unset: an array of them is touched first by the threads that fill it
};
static_assert(sizeof(WideNode) == 128, "WideNode is one 128-B line");

// Wide nodes of a validated SBVH (validateBVH), or an empty vector if the tree cannot have them.
// Node 0 is the root and all its slots are inner: slot i refers to node i + 1 (a leaf or leaf pair
// of the root gets a node of its own), so a kernel needs only the root's boxes. The first
// `topCap` nodes are in breadth-first order, the rest depth first in slot order. Without `loose`, which
// says whether the tree has loose slots, such a tree gets none.
std::vector<WideNode> buildWide(const PhxBVHNode* nodes, uint32_t numNodes, uint32_t topCap,
                                bool* loose = nullptr);

}  // namespace phx
