// Chip-resident time loop, FDORDER 12, viscoelastic P/SV.
#define DN_F 6
#define DN_GROUP 2
#include "dn_resident_inst.inc"
