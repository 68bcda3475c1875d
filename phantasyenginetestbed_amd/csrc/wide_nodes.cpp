// Collapses an SBVH into four-wide nodes; see wide_nodes.hpp.
#include "wide_nodes.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>

namespace phx {
namespace {

// Whether every child box lies within +-2^126 and is not inverted (false for NaN too). `loose` gets a
// flag per node whose child boxes stick out of its own, or stays empty if there are none.
bool eligible(const PhxBVHNode* nodes, uint32_t n, std::vector<uint8_t>& loose)
{
	for (uint32_t i = 0; i < n; i++) {
		const PhxBVHNode& nd = nodes[i];
		for (int c = 0; c < 2; c++) {
			const float* b = nd.fData + 6 * c;
			bool good = true, inside = true;
			for (int k = 0; k < 3; k++)
				good &= std::fabs(b[k]) <= 0x1p126f && std::fabs(b[k + 3]) <= 0x1p126f && b[k] <= b[k + 3];
			if (!good) return false;
			if (nd.iData[2 + c] != 0) continue;
			const float* f = nodes[nd.iData[c]].fData;
			for (int k = 0; k < 3; k++)
				inside &= f[k] >= b[k] && f[k + 6] >= b[k] && f[k + 3] <= b[k + 3] && f[k + 9] <= b[k + 3];
			if (inside) continue;
			if (loose.empty()) loose.resize(n);
			loose[nd.iData[c]] = 1;
		}
	}
	return true;
}

// One slot while a wide node is put together: a leaf, or an inner binary node.
struct Slot {
	const float* box;
	uint32_t ref;    // leaf: the finished reference; inner: the binary node's index
	bool leaf;
	bool loose;      // inner: kWideLoose
	float area;      // half surface area of an inner slot that may be opened, else negative
};

float halfArea(const float* b)
{
	const float x = b[3] - b[0], y = b[4] - b[1], z = b[5] - b[2];
	return x * y + y * z + z * x;
}

// A binary tree, and its loose nodes (none: empty).
struct Tree {
	const PhxBVHNode* nodes;
	std::vector<uint8_t> loose;
	bool isLoose(int32_t node) const { return !loose.empty() && loose[node]; }
};

// Whether a wide node may hold the children of binary node `node` in place of it, whose box is `b`: no ray
// passes a child's box that does not pass b (wide_nodes.hpp: flat boxes), and no child is loose, which has
// to be decided when this node is taken.
bool mayOpen(const Tree& t, int32_t node, const float* b)
{
	const PhxBVHNode& nd = t.nodes[node];
	if (!t.loose.empty())
		for (int c = 0; c < 2; c++)
			if (t.loose[node] || (nd.iData[2 + c] == 0 && t.loose[nd.iData[c]])) return false;
	for (int c = 0; c < 2; c++)
		for (int k = 1; k < 3; k++) {
			const float* f = nd.fData + 6 * c;
			if (f[k] == f[k + 3] && f[k] == b[k + 3] && b[k] < b[k + 3]) return false;
		}
	return true;
}

// The slots of binary node `node` in castRay's order (see wide_nodes.hpp); returns how many (2).
int expand(const Tree& tree, uint32_t node, Slot out[2])
{
	const PhxBVHNode& nd = tree.nodes[node];
	int k = 0;
	for (int c = 0; c < 2; c++)
		if (nd.iData[2 + c] != 0) {
			const uint32_t cnt = uint32_t(nd.iData[2 + c]);
			uint32_t ref = kWideLeaf | uint32_t(~nd.iData[c]) | ((cnt <= 3u ? cnt : 0u) << kWideCountShift);
			if (c == 0 && nd.iData[3] != 0) ref |= kWidePair;
			out[k++] = Slot{nd.fData + 6 * c, ref, true, false, 0.0f};
		}
	for (int c = 1; c >= 0; c--)
		if (nd.iData[2 + c] == 0) {
			const float* b = nd.fData + 6 * c;
			const int32_t at = nd.iData[c];
			out[k++] = Slot{b, uint32_t(at), false, tree.isLoose(at), mayOpen(tree, at, b) ? halfArea(b) : -1.0f};
		}
	return k;
}

// A wide node's slots: binary node `root` with the inner slots of largest area opened in place
// until four are used.
int collapse(const Tree& tree, uint32_t root, Slot s[4])
{
	int k = expand(tree, root, s);
	while (k < 4) {
		int best = -1;
		for (int i = 0; i < k; i++)
			if (!s[i].leaf && s[i].area >= 0.0f && (best < 0 || s[i].area > s[best].area)) best = i;
		if (best < 0) break;
		Slot two[2];
		expand(tree, s[best].ref, two);
		for (int i = k; i > best + 1; i--) s[i] = s[i - 1];
		s[best] = two[0];
		s[best + 1] = two[1];
		k++;
	}
	return k;
}

WideNode emptyNode()
{
	WideNode w;
	const float nan = std::numeric_limits<float>::quiet_NaN();
	for (WideNode::Slot& s : w.slot) s = WideNode::Slot{{nan, nan, nan}, 0u, {nan, nan, nan}, nan};
	return w;
}

void setSlot(WideNode::Slot& s, const float* box, uint32_t ref)
{
	std::memcpy(s.min, box, sizeof(s.min));
	std::memcpy(s.max, box + 3, sizeof(s.max));
	s.ref = ref;
}

}  // namespace

std::vector<WideNode> buildWide(const PhxBVHNode* nodes, uint32_t numNodes, uint32_t topCap, bool* loose)
{
	std::vector<WideNode> out;
	Tree tree{nodes, {}};
	const bool fits = eligible(nodes, numNodes, tree.loose);
	if (loose) *loose = fits && !tree.loose.empty();
	if (!fits || (!loose && !tree.loose.empty())) return out;
	auto inner = [](uint32_t at, bool isLoose) { return at | (isLoose ? kWideLoose : 0u); };

	// A node to fill: the binary node whose subtree it covers and the slots pending beside it.
	struct Item {
		uint32_t at, node, pending;
	};
	std::vector<Item> queue;  // breadth first up to topCap nodes, then a stack
	out.reserve(size_t(numNodes) / 2 + 8);
	out.push_back(emptyNode());
	uint32_t maxPending = 0;

	// The root: its slots become nodes 1..k. Leaves get a node that holds just them.
	Slot s[4];
	const int rootSlots = collapse(tree, 0, s);
	struct RootSlot {
		int first, count;  // range of s
	};
	RootSlot rs[4];
	int numRoot = 0;
	for (int i = 0; i < rootSlots; i++) {
		const int count = s[i].leaf && (s[i].ref & kWidePair) ? 2 : 1;
		rs[numRoot++] = RootSlot{i, count};
		i += count - 1;
	}
	for (int j = 0; j < numRoot; j++) {
		const Slot& a = s[rs[j].first];
		setSlot(out[0].slot[j], a.box, inner(uint32_t(j + 1), a.loose));
		if (rs[j].count == 2) {
			const Slot& b = s[rs[j].first + 1];
			for (int k = 0; k < 3; k++) {
				out[0].slot[j].min[k] = std::min(a.box[k], b.box[k]);
				// (A float more: flat at the maximum, a leaf may be passed by a ray that does not pass there.)
				out[0].slot[j].max[k] = std::nextafter(std::max(a.box[k + 3], b.box[k + 3]), HUGE_VALF);
			}
		}
		out.push_back(emptyNode());
		const uint32_t pending = uint32_t(numRoot - 1 - j);
		if (a.leaf) {
			for (int i = 0; i < rs[j].count; i++)
				setSlot(out[size_t(j) + 1].slot[i], s[rs[j].first + i].box, s[rs[j].first + i].ref);
			maxPending = std::max(maxPending, pending + 1u);
		} else {
			queue.push_back(Item{uint32_t(j + 1), a.ref, pending});
		}
	}
	maxPending = std::max(maxPending, uint32_t(numRoot - 1));

	// Fills node it.at; its inner slots get the next indices and are appended to `next`.
	auto fill = [&](const Item& it, std::vector<Item>& next) {
		Slot t[4];
		const int k = collapse(tree, it.node, t);
		maxPending = std::max(maxPending, it.pending + uint32_t(k - 1));
		for (int i = 0; i < k; i++) {
			if (t[i].leaf) {
				setSlot(out[it.at].slot[i], t[i].box, t[i].ref);
			} else {
				const uint32_t child = uint32_t(out.size());
				setSlot(out[it.at].slot[i], t[i].box, inner(child, t[i].loose));
				out.push_back(emptyNode());
				next.push_back(Item{child, t[i].ref, it.pending + uint32_t(k - 1 - i)});
			}
		}
	};
	size_t head = 0;
	while (head < queue.size() && out.size() < topCap) {
		const Item it = queue[head++];
		fill(it, queue);
	}
	// The rest depth first: a node's children are numbered when it is filled (siblings side by
	// side), the first slot's subtree before the next one's.
	std::vector<Item> stack(queue.rbegin(), queue.rend() - ptrdiff_t(head));
	std::vector<Item> kids;
	while (!stack.empty()) {
		const Item it = stack.back();
		stack.pop_back();
		kids.clear();
		fill(it, kids);
		stack.insert(stack.end(), kids.rbegin(), kids.rend());
	}
	if (maxPending > kWideMaxPending || out.size() > kWideIndex) out.clear();
	for (WideNode& n : out)
		for (int i = 0; i < 3; i++) n.slot[i].lastMax = n.slot[3].max[i];
	return out;
}

}  // namespace phx
